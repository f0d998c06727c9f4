// Symmetric wall-RPY products of a few thousand blobs: the symmetric kernel
// of rmw_wall_rpy.hip on pairs of 64-blob blocks, with the 64 steps of a
// block pair shared by the four waves of a workgroup.
//
// The tile kernel's work item (256 targets x 64 sources or more) is too
// coarse below about ten thousand blobs: 2500 blobs are 220 items for 256 CUs,
// and with one wave per SIMD nothing hides the latency of the dependent
// chains.  Here a work item is a target block I of 64 blobs and a run of
// source blocks J >= I; all four waves hold the same 64 targets (one per
// lane), and wave v takes the steps 16 v .. 16 v + 15 of each block pair, at
// step s lane l meeting source (l + s) mod 64.  2500 blobs are then 820
// workgroups.  The sums of both sides are added over the four waves through
// LDS in a fixed order, so a block pair writes the same partial sums as one
// wave would.  A diagonal block takes the steps 1..32 only: step s and step
// 64 - s are the same pairs (at s = 32 the lower 32 lanes take them).
#include <hip/hip_runtime.h>

#include "rmw_wall_pairs.h"

namespace rmw {

constexpr int kBB = 64;   // blobs per block

template <int MASK, int K, int ACC, typename R, int DOM, bool PER>
__global__ __launch_bounds__(kBlock) void block_kernel(MutParams p)
{
  using BT = BlockTraits<MASK>;
  constexpr int OC = BT::OC, KF = BT::NF ? K : 1, KT = BT::NT ? K : 1;
  static_assert(K <= kBlock / 64, "one staging wave per right-hand side");
  using JT = typename std::conditional<ACC == RMW_PREC_F32_BLOCKED && !PER, float, double>::type;
  // each source twice: the rotated read of step s, entry lane + s, needs no wrap
  __shared__ double s_x[2 * kBB], s_y[2 * kBB], s_z[2 * kBB];
  __shared__ R s_zr[2 * kBB];
  __shared__ R s_f[KF][3][2 * kBB];
  __shared__ R s_t[KT][3][2 * kBB];
  __shared__ double s_sum[kBlock / 64][K][OC][kBB];   // the waves' sums of one side
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  constexpr double pz = DOM == kDomInPlane ? 0.0 : 1.0;   // in plane: P v

  // out[k][l][c] = the four waves' sums, added in order
  auto write_sums = [&](double* out, int cnt) {
    for (int e = threadIdx.x; e < K * kBB * OC; e += kBlock) {
      const int k = e / (kBB * OC), q = e - k * (kBB * OC), l = q / OC, c = q - l * OC;
      if (l < cnt) out[e] = ((s_sum[0][k][c][l] + s_sum[1][k][c][l]) + s_sum[2][k][c][l]) + s_sum[3][k][c][l];
    }
  };

  for (int64_t item = blockIdx.x; item < p.n_items; item += gridDim.x) {
    const MutSys Sy = mut_sys_of_item(p, item);
    const int64_t local = item - Sy.item0;
    const int64_t I = pair_target_tile(local, Sy.n_t, p.chunk_blocks);
    const int64_t J0 = I + (local - items_before(I, Sy.n_t, p.chunk_blocks)) * p.chunk_blocks;
    const int64_t J1 = J0 + p.chunk_blocks < Sy.n_t ? J0 + p.chunk_blocks : Sy.n_t;
    const int icnt = (int)(Sy.n - I * kBB < kBB ? Sy.n - I * kBB : kBB);
    const bool valid = lane < icnt;
    const int64_t gi = Sy.b0 + I * kBB + (valid ? lane : 0);
    // sources are staged by wave: wave v the vectors k = v, v + 4, ... of the
    // 64 sources, the last wave their positions.  The first block's are loaded
    // together with the targets, the following ones a block ahead.
    RawBlob<1, BT::NF, BT::NT> raw;
    auto load_source = [&](int64_t J) {
      const int cnt = (int)(Sy.n - J * kBB < kBB ? Sy.n - J * kBB : kBB);
      const int64_t gj = Sy.b0 + J * kBB + (lane < cnt ? lane : 0);
      const int64_t k = wv < K ? wv : 0;
      if (wv == 3 || wv < K)
        raw.load(p.r, BT::NF ? p.f + k * p.rhs_stride : nullptr, BT::NT ? p.t + k * p.rhs_stride : nullptr, 0, gj);
    };
    load_source(J0);
    double Xi, Yi, Zi, Bi;
    RawBlob<K, BT::NF, BT::NT> own;
    own.load(p.r, p.f, p.t, p.rhs_stride, gi);
    scale_blob(own.r[0], own.r[1], own.r[2], p.a, p.inva, Xi, Yi, Zi, Bi, DOM);
    const R zi = (R)Zi;
    R fi[KF][3], ti[KT][3];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      if constexpr (BT::NF) {
        const double c = valid ? p.c1 * Bi : 0.0;
        fi[k][0] = (R)(c * own.f[k][0]); fi[k][1] = (R)(c * own.f[k][1]); fi[k][2] = (R)(pz * c * own.f[k][2]);
      }
      if constexpr (BT::NT) {
        const double c = valid ? p.c2 * Bi : 0.0;
        ti[k][0] = (R)(c * own.t[k][0]); ti[k][1] = (R)(c * own.t[k][1]); ti[k][2] = (R)(pz * c * own.t[k][2]);
      }
    }
    Acc<ACC> u[K][3], w[K][3];

    for (int64_t J = J0; J < J1; ++J) {
      const int cnt = (int)(Sy.n - J * kBB < kBB ? Sy.n - J * kBB : kBB);
      __syncthreads();   // the previous block (or item) has been consumed
      if (wv == 3 || wv < K) {
        // finite zeros beyond the system (pairs not taken are masked through
        // their geometry)
        const bool in = lane < cnt;
        double X, Y, Z, B;
        scale_blob(raw.r[0], raw.r[1], raw.r[2], p.a, p.inva, X, Y, Z, B, DOM);
        if (wv == 3) {
          X = in ? X : 0.0; Y = in ? Y : 0.0; Z = in ? Z : 0.0;
#pragma unroll
          for (int e = lane; e < 2 * kBB; e += kBB) {
            s_x[e] = X; s_y[e] = Y; s_z[e] = Z; s_zr[e] = (R)Z;
          }
        }
        if (wv < K) {
          auto put = [&](R (&dst)[3][2 * kBB], const double (&v)[3], double c) {
            const R v0 = in ? (R)(c * v[0]) : R(0), v1 = in ? (R)(c * v[1]) : R(0),
                    v2 = in ? (R)(pz * c * v[2]) : R(0);
#pragma unroll
            for (int e = lane; e < 2 * kBB; e += kBB) { dst[0][e] = v0; dst[1][e] = v1; dst[2][e] = v2; }
          };
          if constexpr (BT::NF) put(s_f[wv], raw.f[0], p.c1 * B);
          if constexpr (BT::NT) put(s_t[wv], raw.t[0], p.c2 * B);
        }
      }
      if (J + 1 < J1) load_source(J + 1);
      __syncthreads();
      const bool diag = J == I;
      const bool full = !diag && cnt == kBB && icnt == kBB;
      const int st0 = diag ? 1 + 8 * wv : 16 * wv, st1 = st0 + (diag ? 8 : 16);
      JT ja[K][OC];
#pragma unroll
      for (int k = 0; k < K; ++k)
#pragma unroll
        for (int c = 0; c < OC; ++c) ja[k][c] = JT(0);
      auto steps = [&](auto masked_c) {
        constexpr bool MASKED = decltype(masked_c)::value;
        for (int st = st0; st < st1; ++st) {
          const int jr = lane + st;               // LDS entry of source jr mod 64
          const bool on = !MASKED || (valid && (jr & 63) < cnt && !(diag && st == 32 && lane >= 32));
          const R zj = s_zr[jr];
          auto apply = [&](auto rot_c, R dx, R dy, R dz, auto& sums) {
            mutual_apply<MASK, K, ACC, R, DOM, MASKED, decltype(rot_c)::value>(
                dx, dy, dz, zi, zj, on, fi, ti, [&](int k, int c) { return s_f[BT::NF ? k : 0][c][jr]; },
                [&](int k, int c) { return s_t[BT::NT ? k : 0][c][jr]; }, u, w, sums);
          };
          if constexpr (!PER) {
            apply(std::true_type{}, (R)(Xi - s_x[jr]), (R)(Yi - s_y[jr]), (R)(Zi - s_z[jr]), ja);
          } else {
            ImageSum<ACC, R> ji[K][OC];
#pragma unroll
            for (int k = 0; k < K; ++k)
#pragma unroll
              for (int c = 0; c < OC; ++c) ji[k][c] = 0;
            each_image<R>(Xi - s_x[jr], Yi - s_y[jr], Zi - s_z[jr], p.periodic, p.L, p.iL,
                          [&](R dx, R dy, R dz, bool) { apply(std::false_type{}, dx, dy, dz, ji); });
#pragma unroll
            for (int k = 0; k < K; ++k)
#pragma unroll
              for (int c = 0; c < OC; ++c) ja[k][c] = rol1(ja[k][c]) + (JT)ji[k][c];
            flush_all<K, ACC>(u, w);
          }
        }
      };
      // full off-diagonal block pairs run without masks (single outputs only:
      // a second copy of the four-block loop costs registers)
      if constexpr (OC == 3 && K == 1) {
        if (full) steps(std::false_type{}); else steps(std::true_type{});
      } else {
        steps(std::true_type{});
      }
      flush_all<K, ACC>(u, w);   // at most kSub sources since the last fold
      const int jw = (lane + st1 - 1) & 63;   // the source whose sum this lane holds
#pragma unroll
      for (int k = 0; k < K; ++k)
#pragma unroll
        for (int c = 0; c < OC; ++c) s_sum[wv][k][c][jw] = (double)ja[k][c];
      __syncthreads();
      write_sums(p.part_j + (Sy.pj0 + tri_index(J, I)) * (K * kBB * OC), cnt);
    }
    __syncthreads();   // the last block's source-side sums have been written out
#pragma unroll
    for (int k = 0; k < K; ++k) {
      if constexpr (BT::HU) {
#pragma unroll
        for (int c = 0; c < 3; ++c) s_sum[wv][k][c][lane] = u[k][c].get();
      }
      if constexpr (BT::HW) {
        constexpr int o = BT::HU ? 3 : 0;
#pragma unroll
        for (int c = 0; c < 3; ++c) s_sum[wv][k][o + c][lane] = w[k][c].get();
      }
    }
    __syncthreads();
    write_sums(p.part_i + (Sy.pi0 + local) * (K * kBB * OC), icnt);
  }
}

template <int MASK, int K, int DOM, bool PER>
static void launch_prec(int prec, const MutParams& q, int grid, hipStream_t st)
{
  const dim3 g(grid), b(kBlock);
  if (prec == RMW_PREC_F32_BLOCKED)
    hipLaunchKernelGGL((block_kernel<MASK, K, RMW_PREC_F32_BLOCKED, float, DOM, PER>), g, b, 0, st, q);
  else if (prec == RMW_PREC_F32_F64ACC)
    hipLaunchKernelGGL((block_kernel<MASK, K, RMW_PREC_F32_F64ACC, float, DOM, PER>), g, b, 0, st, q);
  else if (prec == RMW_PREC_F32_KAHAN)
    hipLaunchKernelGGL((block_kernel<MASK, K, RMW_PREC_F32_KAHAN, float, DOM, PER>), g, b, 0, st, q);
  else
    hipLaunchKernelGGL((block_kernel<MASK, K, RMW_PREC_F64, double, DOM, PER>), g, b, 0, st, q);
}

template <int MASK>
static void launch_wall(int prec, int K, const MutParams& q, int grid, hipStream_t st)
{
  if (q.periodic) return launch_prec<MASK, 1, kDomWall, true>(prec, q, grid, st);
  if constexpr (MASK == kUF || MASK == 15) {
    if (K == 4) return launch_prec<MASK, 4, kDomWall, false>(prec, q, grid, st);
    if (K == 2) return launch_prec<MASK, 2, kDomWall, false>(prec, q, grid, st);
  }
  launch_prec<MASK, 1, kDomWall, false>(prec, q, grid, st);
}

void launch_blocks(int domain, int mask, int prec, int K, const MutParams& q, int grid, hipStream_t st)
{
  if (domain == kDomWall) {
    switch (mask) {
      case 1: return launch_wall<1>(prec, K, q, grid, st);
      case 2: return launch_wall<2>(prec, K, q, grid, st);
      case 3: return launch_wall<3>(prec, K, q, grid, st);
      case 4: return launch_wall<4>(prec, K, q, grid, st);
      case 8: return launch_wall<8>(prec, K, q, grid, st);
      default: return launch_wall<15>(prec, K, q, grid, st);
    }
  }
  if (domain == kDomNoWall) {
    switch (mask) {
      case 1: return launch_prec<1, 1, kDomNoWall, false>(prec, q, grid, st);
      case 2: return launch_prec<2, 1, kDomNoWall, false>(prec, q, grid, st);
      case 3: return launch_prec<3, 1, kDomNoWall, false>(prec, q, grid, st);
      case 4: return launch_prec<4, 1, kDomNoWall, false>(prec, q, grid, st);
      case 8: return launch_prec<8, 1, kDomNoWall, false>(prec, q, grid, st);
      default: return launch_prec<15, 1, kDomNoWall, false>(prec, q, grid, st);
    }
  }
  if (domain == kDomFreeSurface) return launch_prec<1, 1, kDomFreeSurface, false>(prec, q, grid, st);
  switch (mask) {
    case 1: return launch_prec<1, 1, kDomInPlane, false>(prec, q, grid, st);
    case 2: return launch_prec<2, 1, kDomInPlane, false>(prec, q, grid, st);
    default: return launch_prec<3, 1, kDomInPlane, false>(prec, q, grid, st);
  }
}

}  // namespace rmw
