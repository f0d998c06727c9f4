// Wall-RPY products of few blobs in one launch.
//
// With a few hundred blobs the two-launch kernels leave the chip idle: 172
// blobs are one 256-target tile, so one workgroup walked all the sources
// serially, and the partial sums needed a second launch.  Here a workgroup
// owns TT targets and its 256 threads share the sources: thread t takes the
// sources t, t + 256, ... and evaluates each against all TT targets (whose
// positions are uniform over the workgroup: TT independent dependency chains
// per wave), so n blobs occupy n / TT workgroups.  The 256 partial sums per
// output are added through LDS in a fixed order and the self term, damping
// and scaling applied in place: no partial sums in memory, no second
// launch.  Every ordered pair is evaluated, twice the work of the symmetric
// kernels, which is why the rule in rmw_wall_rpy.hip (direct_pairs) stops
// using it where those win.
#include <hip/hip_runtime.h>

#include "rmw_wall_pairs.h"

namespace rmw {

// Targets per workgroup: a loaded source serves that many pairs; at most 24
// running sums per thread.
constexpr int targets_of(int oc, int K) { return oc * K <= 6 ? 4 : (oc * K <= 12 ? 2 : 1); }

template <int MASK, int K, int ACC, typename R, int DOM, bool PER>
__global__ __launch_bounds__(kBlock) void direct_kernel(DirectParams p)
{
  using BT = BlockTraits<MASK>;
  constexpr int OC = BT::OC, TT = targets_of(OC, K);
  constexpr int V = TT * K * OC;
  // 16 outputs are reduced at a time, 16 threads each; rows padded so that
  // four rows' reads fall into different banks
  constexpr int kRow = kBlock + 16;
  __shared__ double s_part[V < 16 ? V : 16][kRow];

  DirectSys S = p.single;
  if (p.table) {
    int lo = 0, hi = p.nsys - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (p.table[mid].item0 <= (int64_t)blockIdx.x) lo = mid; else hi = mid - 1;
    }
    S = p.table[lo];
  }
  const int64_t t0 = ((int64_t)blockIdx.x - S.item0) * TT;
  double Xi[TT], Yi[TT], Zi[TT], Bi;
  R zi[TT];
#pragma unroll
  for (int q = 0; q < TT; ++q) {
    // targets beyond the system repeat its last blob; their sums are dropped
    const int64_t il = t0 + q < S.n ? t0 + q : S.n - 1;
    load_blob(p.r, S.b0 + il, p.a, p.inva, Xi[q], Yi[q], Zi[q], Bi, DOM);
    zi[q] = (R)Zi[q];
  }
  Acc<ACC> u[TT][K][3], w[TT][K][3];
  constexpr double pz = DOM == kDomInPlane ? 0.0 : 1.0;   // in plane: P v

  int taken = 0;
  RawBlob<K, BT::NF, BT::NT> raw;   // the next source, loaded a step ahead
  raw.load(p.r, p.f, p.t, p.rhs_stride, S.b0 + ((int64_t)threadIdx.x < S.n ? threadIdx.x : 0));
  for (int64_t j = threadIdx.x; j < S.n; j += kBlock) {
    double X, Y, Z, B;
    scale_blob(raw.r[0], raw.r[1], raw.r[2], p.a, p.inva, X, Y, Z, B, DOM);
    const R zj = (R)Z;
    Vec3<R> fv[BT::NF ? K : 1], tv[BT::NT ? K : 1];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      if constexpr (BT::NF) {
        const double c = p.c1 * B;
        fv[k] = Vec3<R>{(R)(c * raw.f[k][0]), (R)(c * raw.f[k][1]), (R)(pz * c * raw.f[k][2])};
      }
      if constexpr (BT::NT) {
        const double c = p.c2 * B;
        tv[k] = Vec3<R>{(R)(c * raw.t[k][0]), (R)(c * raw.t[k][1]), (R)(pz * c * raw.t[k][2])};
      }
    }
    if (j + kBlock < S.n) raw.load(p.r, p.f, p.t, p.rhs_stride, S.b0 + j + kBlock);
    auto sf = [&](int k) { return fv[BT::NF ? k : 0]; };
    auto st = [&](int k) { return tv[BT::NT ? k : 0]; };
    ++taken;
#pragma unroll
    for (int q = 0; q < TT; ++q) {
      const bool own = j == t0 + q;
      if constexpr (!PER) {
        pair_eval<MASK, K, ACC, R, DOM>((R)(Xi[q] - X), (R)(Yi[q] - Y), (R)(Zi[q] - Z), zi[q], zj, sf, st, own,
                                        u[q], w[q]);
      } else {
        each_image<R>(Xi[q] - X, Yi[q] - Y, Zi[q] - Z, p.periodic, p.L, p.iL,
                      [&](R dx, R dy, R dz, bool central) {
                        pair_eval<MASK, K, ACC, R, DOM>(dx, dy, dz, zi[q], zj, sf, st, own && central, u[q], w[q]);
                      });
      }
    }
    // fold the FP32 sums every kSub sources (every source with the images)
    if (PER || (taken & (kSub - 1)) == 0) {
#pragma unroll
      for (int q = 0; q < TT; ++q) flush_all<K, ACC>(u[q], w[q]);
    }
  }

  // value (q K + k) OC + c: output c of right-hand side k of target q
  const int row = threadIdx.x >> 4, sub = threadIdx.x & 15;
#pragma unroll
  for (int o0 = 0; o0 < V; o0 += 16) {
    if (o0 > 0) __syncthreads();   // the previous 16 outputs have been read
#pragma unroll
    for (int o = o0; o < V && o < o0 + 16; ++o) {
      const int q = o / (K * OC), k = (o / OC) % K, c = o % OC;
      const bool is_w = BT::HW && (!BT::HU || c >= 3);
      s_part[o - o0][threadIdx.x] = is_w ? w[q][k][c % 3].get() : u[q][k][c % 3].get();
    }
    __syncthreads();
    const int o = o0 + row;
    if (o < V) {
      double s = 0.0;
#pragma unroll
      for (int m = 0; m < kBlock / 16; ++m) s += s_part[row][sub + 16 * m];
#pragma unroll
      for (int m = 8; m >= 1; m >>= 1) s += __shfl_xor(s, m, 16);
      const int q = o / (K * OC), k = (o / OC) % K, c = o % OC;
      if (sub == 0 && t0 + q < S.n)
        finish_output(p.r, p.f, p.t, p.vel, p.omg, MASK, k, S.b0 + t0 + q, c, s, p.rhs_stride, p.out_stride, p.a,
                      p.inva, p.c1, p.c2, DOM);
    }
  }
}

template <int MASK, int K, int DOM, bool PER>
static void launch_prec(int prec, const DirectParams& q, dim3 g, hipStream_t st)
{
  const dim3 b(kBlock);
  if (prec == RMW_PREC_F32_BLOCKED)
    hipLaunchKernelGGL((direct_kernel<MASK, K, RMW_PREC_F32_BLOCKED, float, DOM, PER>), g, b, 0, st, q);
  else if (prec == RMW_PREC_F32_F64ACC)
    hipLaunchKernelGGL((direct_kernel<MASK, K, RMW_PREC_F32_F64ACC, float, DOM, PER>), g, b, 0, st, q);
  else if (prec == RMW_PREC_F32_KAHAN)
    hipLaunchKernelGGL((direct_kernel<MASK, K, RMW_PREC_F32_KAHAN, float, DOM, PER>), g, b, 0, st, q);
  else
    hipLaunchKernelGGL((direct_kernel<MASK, K, RMW_PREC_F64, double, DOM, PER>), g, b, 0, st, q);
}

template <int MASK, int K, int DOM>
static void launch_per(int prec, const DirectParams& q, dim3 g, hipStream_t st)
{
  if (q.periodic) launch_prec<MASK, K, DOM, true>(prec, q, g, st);
  else launch_prec<MASK, K, DOM, false>(prec, q, g, st);
}

template <int DOM>
static void launch_mask(int mask, int prec, const DirectParams& q, dim3 g, hipStream_t st)
{
  switch (mask) {
    case 1: return launch_per<1, 1, DOM>(prec, q, g, st);
    case 2: return launch_per<2, 1, DOM>(prec, q, g, st);
    case 3: return launch_per<3, 1, DOM>(prec, q, g, st);
    case 4: return launch_per<4, 1, DOM>(prec, q, g, st);
    case 5: return launch_per<5, 1, DOM>(prec, q, g, st);
    case 8: return launch_per<8, 1, DOM>(prec, q, g, st);
    case 10: return launch_per<10, 1, DOM>(prec, q, g, st);
    case 12: return launch_per<12, 1, DOM>(prec, q, g, st);
    default: return launch_per<15, 1, DOM>(prec, q, g, st);
  }
}

int direct_targets(int mask, int K)
{
  const int oc = ((mask & (kUF | kUT)) ? 3 : 0) + ((mask & (kWF | kWT)) ? 3 : 0);
  return targets_of(oc, K);
}

// Several right-hand sides share a launch for the products the solvers
// take with several (UF and all four blocks above the wall).
int direct_max_k(int mask, int domain)
{
  return domain == kDomWall && (mask == kUF || mask == (kUF | kUT | kWF | kWT)) ? 4 : 1;
}

void launch_direct(int domain, int mask, int prec, int K, const DirectParams& q, int64_t wgs, hipStream_t st)
{
  const dim3 g((unsigned)wgs);
  if (K > 1) {
    if (mask == kUF) {
      if (K == 4) launch_per<kUF, 4, kDomWall>(prec, q, g, st);
      else launch_per<kUF, 2, kDomWall>(prec, q, g, st);
    } else {
      if (K == 4) launch_per<15, 4, kDomWall>(prec, q, g, st);
      else launch_per<15, 2, kDomWall>(prec, q, g, st);
    }
    return;
  }
  if (domain == kDomWall) return launch_mask<kDomWall>(mask, prec, q, g, st);
  if (domain == kDomNoWall) return launch_mask<kDomNoWall>(mask, prec, q, g, st);
  if (domain == kDomFreeSurface) return launch_per<kUF, 1, kDomFreeSurface>(prec, q, g, st);
  switch (mask) {
    case 1: return launch_per<1, 1, kDomInPlane>(prec, q, g, st);
    case 2: return launch_per<2, 1, kDomInPlane>(prec, q, g, st);
    default: return launch_per<3, 1, kDomInPlane>(prec, q, g, st);
  }
}

}  // namespace rmw
