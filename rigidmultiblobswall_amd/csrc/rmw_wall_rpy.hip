// Wall-corrected RPY blob mobility products on gfx950 (MI355X).
//
// One call evaluates any subset of the grand mobility blocks
// [[UF, UT], [WF, WT]] for k right-hand sides on one suspension, or on a
// ragged batch of independent suspensions.  Few blobs take one launch
// (rmw_wall_direct.hip), up to some thousand the symmetric kernel on 64-blob
// blocks (rmw_wall_blocks.hip), larger suspensions the symmetric kernel on
// 256-blob tiles below (section 3b), each followed by one reduce; what those
// do not serve, or a tuning that asks for it, runs the ordered kernels in two
// launches:
//
//   1. pair   : all-pairs sums; each workgroup owns 256 targets (one per
//               lane, in registers) and one chunk of sources that it
//               streams through LDS in tiles of 256, reading positions and
//               sources straight from the caller's float64 arrays: z_eff =
//               max(z, a), damping B = min(z/a, 1) and 1/(8 pi eta a^p) are
//               applied as a tile is staged.  The RPY and wall image terms
//               are fused in one pass and the geometry is shared by all
//               blocks and right-hand sides.  Partial sums (FP64) go to the
//               workspace, one slot per (chunk, target).
//   2. reduce : fixed-order FP64 sum over chunks, FP64 self term, B and
//               the remaining 1/a factor, written as (k, n, 3) float64.
//
// Reference: mobility/mobility_numba.py:123-287 (UF), :547-686 (UT),
// :937-1073 (WF), :1188-1328 (WT); wrappers mobility/mobility.py:52-84,
// 1132-1342; pseudo-periodic images mobility_numba.py:149-198.
//
// FP32 modes.  Subtracting two FP32 coordinates of size X loses ~6e-8 X of
// absolute accuracy, which for near pairs (|d| ~ a, X up to ~500 a) would be
// a 3e-5 relative error.  The difference d = r_i - r_j (and its periodic
// shifts) is therefore formed in FP64 and rounded once to FP32, so d
// carries FP32 relative accuracy in d itself; everything after that is
// FP32.  (On gfx950 an FP64 add issues at the rate of an unpacked FP32 add.)
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <type_traits>
#include <vector>

#include "rmw_wall_pairs.h"

namespace rmw {

// ---------------------------------------------------------------------------
// Errors and device properties
// ---------------------------------------------------------------------------
static thread_local std::string g_last_error;
void set_last_error(const std::string& msg) { g_last_error = msg; }

const DeviceProps& device_props()
{
  static std::mutex mu;
  static DeviceProps cache[64];
  int dev = 0;
  RMW_CHECK_HIP(hipGetDevice(&dev));
  RMW_REQUIRE(dev >= 0 && dev < 64, "device ordinal out of range");
  std::lock_guard<std::mutex> lk(mu);
  DeviceProps& p = cache[dev];
  if (p.device < 0) {
    hipDeviceProp_t prop;
    RMW_CHECK_HIP(hipGetDeviceProperties(&prop, dev));
    p.cu_count = prop.multiProcessorCount;
    p.clock_khz = prop.clockRate;
    p.warp = prop.warpSize;
    p.arch = prop.gcnArchName;
    p.device = dev;
  }
  return p;
}

// One independent suspension of the batch and its share of the work list.
struct SysInfo {
  int64_t b0;         // first blob (global index)
  int64_t n;          // blobs
  int64_t n_tt;       // target tiles of kBlock
  int64_t n_chunks;   // source chunks
  int64_t chunk_len;  // sources per chunk (multiple of kBlock)
  int64_t item0;      // first work item
  int64_t part0;      // first partial (in doubles)
};

struct PairParams {
  const double* r;        // (ntot, 3) positions
  const double* f;        // K right-hand sides rhs_stride apart, or null
  const double* t;
  int64_t rhs_stride;
  double a, inva, c1, c2; // c1 = 1/(8 pi eta a), c2 = c1 / a
  double* partial;
  const SysInfo* table;   // nullptr -> single
  SysInfo single;
  int nsys;
  int64_t ntot;
  int64_t total_items;
  int periodic;           // bit d set when L_d > 0
  double L[3], iL[3];     // periodic lengths / a and their inverses (0: none)
  int domain;             // kDomWall, kDomNoWall, kDomInPlane, kDomFreeSurface
};

__device__ inline SysInfo find_sys_item(const PairParams& p, int64_t item)
{
  if (!p.table) return p.single;
  int lo = 0, hi = p.nsys - 1;
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if (p.table[mid].item0 <= item) lo = mid; else hi = mid - 1;
  }
  return p.table[lo];
}

// Source record of the FP32 kernels: FP64 position for the difference, FP32
// height for the wall terms (two 16-byte LDS reads).
struct __align__(16) SrcF32 {
  double x, y, z;
  float zf, pad;
};

// ---------------------------------------------------------------------------
// 3. pair kernels
// ---------------------------------------------------------------------------
// Per-target accumulator policies: rmw_accum.h.

// Partial sums of one work item: slot (chunk, rhs, target) of the system.
template <int MASK, int K, typename A>
__device__ __forceinline__ void store_partials(const PairParams& p, const SysInfo& S, int64_t ch, int64_t il,
                                               A (&u)[K][3], A (&w)[K][3])
{
  using BT = BlockTraits<MASK>;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    double* P = p.partial + S.part0 + ((ch * K + k) * S.n + il) * BT::OC;
    int o = 0;
    if constexpr (BT::HU) {
      P[0] = u[k][0].get(); P[1] = u[k][1].get(); P[2] = u[k][2].get();
      o = 3;
    }
    if constexpr (BT::HW) {
      P[o] = w[k][0].get(); P[o + 1] = w[k][1].get(); P[o + 2] = w[k][2].get();
    }
  }
}

template <typename V> __device__ V make_v4(double x, double y, double z);
template <> __device__ __forceinline__ float4 make_v4<float4>(double x, double y, double z)
{
  return make_float4((float)x, (float)y, (float)z, 0.0f);
}
template <> __device__ __forceinline__ double4 make_v4<double4>(double x, double y, double z)
{
  return make_double4(x, y, z, 0.0);
}

// Stage the sources of blob gj for K right-hand sides into LDS slot `slot`:
// B f / (8 pi eta a) and B t / (8 pi eta a^2) as float4 or double4.
template <int MASK, int K, typename V, int DOM>
__device__ __forceinline__ void stage_sources(const PairParams& p, int64_t gj, double B, int slot, V* s_f, V* s_t)
{
  using BT = BlockTraits<MASK>;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    // in plane: only the x-y components act (P v)
    const double pz = DOM == kDomInPlane ? 0.0 : 1.0;
    if constexpr (BT::NF) {
      const double* v = p.f + k * p.rhs_stride + 3 * gj;
      const double c = p.c1 * B;
      s_f[k * kBlock + slot] = make_v4<V>(c * v[0], c * v[1], pz * c * v[2]);
    }
    if constexpr (BT::NT) {
      const double* v = p.t + k * p.rhs_stride + 3 * gj;
      const double c = p.c2 * B;
      s_t[k * kBlock + slot] = make_v4<V>(c * v[0], c * v[1], pz * c * v[2]);
    }
  }
}

// Source j of right-hand side k in the ordered kernels' LDS arrays.
template <typename V>
__device__ __forceinline__ auto lds(const V* __restrict__ s, int j)
{
  return [=](int k) { return s[k * kBlock + j]; };
}

// Minimum resident waves per SIMD asked of the register allocator for the
// FP32 pair kernels (1 = no constraint).
#ifndef RMW_PAIR_WAVES
#define RMW_PAIR_WAVES 1
#endif
template <int MASK, int K>
constexpr int pair_min_waves()
{
  return (K == 1 && (MASK == kUF || MASK == kUT || MASK == kWF || MASK == kWT)) ? RMW_PAIR_WAVES : 1;
}

template <int MASK, int K, int ACC, int DOM = kDomWall>
__global__ __launch_bounds__(kBlock, (pair_min_waves<MASK, K>())) void pair_kernel_f32(PairParams p)
{
  using BT = BlockTraits<MASK>;
  __shared__ SrcF32 s_pos[kBlock];
  __shared__ float4 s_f[BT::NF ? K * kBlock : 1];
  __shared__ float4 s_t[BT::NT ? K * kBlock : 1];

  for (int64_t item = blockIdx.x; item < p.total_items; item += gridDim.x) {
    const SysInfo S = find_sys_item(p, item);
    const int64_t local = item - S.item0;
    const int64_t tt = local / S.n_chunks;
    const int64_t ch = local - tt * S.n_chunks;
    const int64_t t0 = tt * kBlock;
    const int64_t il = t0 + threadIdx.x;
    const bool valid = il < S.n;
    double Xi, Yi, Zi, Bi;
    load_blob(p.r, S.b0 + (valid ? il : 0), p.a, p.inva, Xi, Yi, Zi, Bi, DOM);
    const float zi = (float)Zi;

    Acc<ACC> u[K][3], w[K][3];

    const int64_t s_begin = ch * S.chunk_len;
    const int64_t s_end = s_begin + S.chunk_len < S.n ? s_begin + S.chunk_len : S.n;
    for (int64_t s0 = s_begin; s0 < s_end; s0 += kBlock) {
      const int cnt = (int)(s_end - s0 < kBlock ? s_end - s0 : kBlock);
      __syncthreads();  // the previous tile has been consumed
      if ((int)threadIdx.x < cnt) {
        const int64_t gj = S.b0 + s0 + threadIdx.x;
        double X, Y, Z, B;
        load_blob(p.r, gj, p.a, p.inva, X, Y, Z, B, DOM);
        s_pos[threadIdx.x] = SrcF32{X, Y, Z, (float)Z, 0.0f};
        stage_sources<MASK, K, float4, DOM>(p, gj, B, threadIdx.x, s_f, s_t);
      }
      __syncthreads();
      // Tiles that contain this workgroup's own targets need the self mask.
      const bool diag = (s0 < t0 + kBlock) && (t0 < s0 + cnt);
      const int self_j = (int)(il - s0);  // local source index of the target itself
      if (!p.periodic) {
        auto eval = [&](int j, bool masked) {
          const SrcF32 sp = s_pos[j];
          const float dx = (float)(Xi - sp.x);
          const float dy = (float)(Yi - sp.y);
          const float dz = (float)(Zi - sp.z);
          pair_eval<MASK, K, ACC, float, DOM>(dx, dy, dz, zi, sp.zf, lds(s_f, j), lds(s_t, j),
                                              masked && j == self_j, u, w);
        };
        int j = 0;
        if (diag) {
          for (; j + kSub <= cnt; j += kSub) {
#pragma unroll 2
            for (int jj = 0; jj < kSub; ++jj) eval(j + jj, true);
            flush_all<K, ACC>(u, w);
          }
          for (; j < cnt; ++j) eval(j, true);
        } else {
          for (; j + kSub <= cnt; j += kSub) {
#pragma unroll 2
            for (int jj = 0; jj < kSub; ++jj) eval(j + jj, false);
            flush_all<K, ACC>(u, w);
          }
          for (; j < cnt; ++j) eval(j, false);
        }
        flush_all<K, ACC>(u, w);
      } else {
        for (int j = 0; j < cnt; ++j) {
          const SrcF32 sp = s_pos[j];
          each_image<float>(Xi - sp.x, Yi - sp.y, Zi - sp.z, p.periodic, p.L, p.iL,
                            [&](float dx, float dy, float dz, bool central) {
                              pair_eval<MASK, K, ACC, float, DOM>(dx, dy, dz, zi, sp.zf, lds(s_f, j), lds(s_t, j),
                                                                  diag && central && (j == self_j), u, w);
                            });
          flush_all<K, ACC>(u, w);
        }
      }
    }
    if (valid) store_partials<MASK, K>(p, S, ch, il, u, w);
  }
}

template <int MASK, int K, int DOM = kDomWall>
__global__ __launch_bounds__(kBlock) void pair_kernel_f64(PairParams p)
{
  using BT = BlockTraits<MASK>;
  __shared__ double4 s_pos[kBlock];
  __shared__ double4 s_f[BT::NF ? K * kBlock : 1];
  __shared__ double4 s_t[BT::NT ? K * kBlock : 1];

  for (int64_t item = blockIdx.x; item < p.total_items; item += gridDim.x) {
    const SysInfo S = find_sys_item(p, item);
    const int64_t local = item - S.item0;
    const int64_t tt = local / S.n_chunks;
    const int64_t ch = local - tt * S.n_chunks;
    const int64_t t0 = tt * kBlock;
    const int64_t il = t0 + threadIdx.x;
    const bool valid = il < S.n;
    double Xi, Yi, Zi, Bi;
    load_blob(p.r, S.b0 + (valid ? il : 0), p.a, p.inva, Xi, Yi, Zi, Bi, DOM);

    Acc<RMW_PREC_F64> u[K][3], w[K][3];
    const int64_t s_begin = ch * S.chunk_len;
    const int64_t s_end = s_begin + S.chunk_len < S.n ? s_begin + S.chunk_len : S.n;
    for (int64_t s0 = s_begin; s0 < s_end; s0 += kBlock) {
      const int cnt = (int)(s_end - s0 < kBlock ? s_end - s0 : kBlock);
      __syncthreads();
      if ((int)threadIdx.x < cnt) {
        const int64_t gj = S.b0 + s0 + threadIdx.x;
        double X, Y, Z, B;
        load_blob(p.r, gj, p.a, p.inva, X, Y, Z, B, DOM);
        s_pos[threadIdx.x] = make_double4(X, Y, Z, 0.0);
        stage_sources<MASK, K, double4, DOM>(p, gj, B, threadIdx.x, s_f, s_t);
      }
      __syncthreads();
      const bool diag = (s0 < t0 + kBlock) && (t0 < s0 + cnt);
      const int self_j = (int)(il - s0);
      for (int j = 0; j < cnt; ++j) {
        const double4 pj = s_pos[j];
        double rx = Xi - pj.x, ry = Yi - pj.y, rz = Zi - pj.z;
        if (!p.periodic) {
          pair_eval<MASK, K, RMW_PREC_F64, double, DOM>(rx, ry, rz, Zi, pj.z, lds(s_f, j), lds(s_t, j),
                                                        diag && j == self_j, u, w);
        } else {
          each_image<double>(rx, ry, rz, p.periodic, p.L, p.iL, [&](double dx, double dy, double dz, bool central) {
            pair_eval<MASK, K, RMW_PREC_F64, double, DOM>(dx, dy, dz, Zi, pj.z, lds(s_f, j), lds(s_t, j),
                                                          diag && central && (j == self_j), u, w);
          });
        }
      }
    }
    if (valid) store_partials<MASK, K>(p, S, ch, il, u, w);
  }
}

// ---------------------------------------------------------------------------
// 3b. symmetric ("mutual") kernels.  The wall mobility is symmetric:
//     UF_ji = UF_ij^T, WT_ji = WT_ij^T, UT_ji = WF_ij^T, WF_ji = UT_ij^T, so
//     each unordered pair is evaluated once and serves both blobs.  Work
//     items are (target tile T, run of source tiles S >= T) of one system.
//     Each wave owns 64 targets (registers) and sweeps a source tile in
//     blocks of 64: at step s lane l takes source (l + s) mod 64 of the
//     block, so the 64 lanes touch 64 different sources (structure-of-arrays
//     LDS, conflict-free).  The source-side sum of a source travels with it:
//     every step the accumulator register moves one lane down (DPP
//     wave_rol:1, fused into the add), so after the 64 steps each source's
//     sum over the wave's targets sits in one lane.  After each block the
//     four waves' sums are added in a fixed order.  On the diagonal tile
//     (S == T) only sources above the target are taken.  Partial sums: one
//     slot per item (target side) and one per tile pair (S, T) (source side),
//     reduced in a fixed order.
// ---------------------------------------------------------------------------
// Largest workspace the automatic choice gives the symmetric kernels.
constexpr size_t kMutAutoBytes = size_t(2) << 30;

// Symmetric pair kernel.  R = float: FP32 pair terms (ACC: the target-side
// accumulator; source side: FP32 sums over 16 steps folded into FP64 in the
// blocked mode, an FP64 travelling accumulator otherwise); R = double: FP64.
// PER: pseudo-periodic images (mobility_numba.py:149-198).  The minimum
// image is odd in d and the box set {-1, 0, 1} is symmetric, so the images
// of (j, i) are the negated images of (i, j) and M_ji = M_ij^T holds image
// by image; each unordered pair takes all its images on both sides, sums
// are folded every step, and the self pair's images outside the central box
// are added by the reduce.
template <int MASK, int K, int ACC, typename R, int DOM = kDomWall, bool PER = false>
__global__ __launch_bounds__(kBlock) void mutual_kernel(MutParams p)
{
  using BT = BlockTraits<MASK>;
  constexpr bool UF = (MASK & kUF) != 0, UT = (MASK & kUT) != 0, WF = (MASK & kWF) != 0, WT = (MASK & kWT) != 0;
  constexpr int OC = BT::OC;
  constexpr bool kFoldJ = ACC == RMW_PREC_F32_BLOCKED && !PER;
  // several right-hand sides: form each pair's blocks once as 3x3 matrices
  constexpr bool kMat = K >= 2;
  using JT = typename std::conditional<kFoldJ, float, double>::type;
  // single-output kernels of one right-hand side store each 64-source
  // block twice (entry 128 b + m, m < 128, holds source 64 b + m mod 64), so
  // the rotated read of step s, entry 128 b + lane + s, needs no wrap
  // (1.5 % faster UF product at 32768 blobs; not for the two-output kernel)
  constexpr bool kDbl = !kMat && !PER && OC == 3;
  constexpr int kLds = kDbl ? 2 * kBlock : kBlock;
  __shared__ double s_x[kLds], s_y[kLds], s_z[kLds];
  __shared__ R s_zr[kLds];
  __shared__ R s_f[BT::NF ? K : 1][3][kLds];
  __shared__ R s_t[BT::NT ? K : 1][3][kLds];
  __shared__ double s_jd[kBlock / 64][K][OC][64];  // per-wave source-side sums of one block
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int il = threadIdx.x;
  // fold the FP32 sums every kSub sources (every source with the images)
  constexpr int kFold = PER ? 0 : kSub - 1;

  for (int64_t item = blockIdx.x; item < p.n_items; item += gridDim.x) {
    const MutSys Sy = mut_sys_of_item(p, item);
    const int64_t local = item - Sy.item0;
    const int64_t T = pair_target_tile_blocks(local, Sy.n_t, p.chunk_blocks);
    const int64_t blk0 = 4 * T + (local - items_before_blocks(T, Sy.n_t, p.chunk_blocks)) * p.chunk_blocks;
    const int64_t blk1 = blk0 + p.chunk_blocks < 4 * Sy.n_t ? blk0 + p.chunk_blocks : 4 * Sy.n_t;
    const int64_t S0 = blk0 >> 2, S1 = (blk1 + 3) >> 2;
    const int64_t i = T * kBlock + il;  // within the system
    const bool valid = i < Sy.n;
    const int64_t gi = Sy.b0 + (valid ? i : 0);
    double Xi, Yi, Zi, Bi;
    load_blob(p.r, gi, p.a, p.inva, Xi, Yi, Zi, Bi, DOM);
    constexpr double pz = DOM == kDomInPlane ? 0.0 : 1.0;   // in plane: P v
    const R zi = (R)Zi;
    R fi[BT::NF ? K : 1][3], ti[BT::NT ? K : 1][3];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      if constexpr (BT::NF) {
        const double* v = p.f + k * p.rhs_stride + 3 * gi;
        const double c = valid ? p.c1 * Bi : 0.0;
        fi[k][0] = (R)(c * v[0]); fi[k][1] = (R)(c * v[1]); fi[k][2] = (R)(pz * c * v[2]);
      }
      if constexpr (BT::NT) {
        const double* v = p.t + k * p.rhs_stride + 3 * gi;
        const double c = valid ? p.c2 * Bi : 0.0;
        ti[k][0] = (R)(c * v[0]); ti[k][1] = (R)(c * v[1]); ti[k][2] = (R)(pz * c * v[2]);
      }
    }
    Acc<ACC> u[K][3], w[K][3];

    for (int64_t S = S0; S < S1; ++S) {
      const int64_t s0 = S * kBlock;
      const int cnt = (int)(Sy.n - s0 < kBlock ? Sy.n - s0 : kBlock);
      // the 64-source blocks of this tile the item covers: only their
      // sources are staged (an item of one block reads a quarter of the tile)
      const int bb0 = S == S0 ? (int)(blk0 - 4 * S) : 0;
      const int bb1 = blk1 - 4 * S < kBlock / 64 ? (int)(blk1 - 4 * S) : kBlock / 64;
      __syncthreads();  // the previous tile has been consumed
      if ((il >> 6) >= bb0 && (il >> 6) < bb1) {
        // the source record of this thread (finite zeros beyond the system:
        // pairs not taken are masked through their geometry, make_geom_on,
        // and still multiply these values by zero coefficients)
        double X = 0.0, Y = 0.0, Z = 0.0;
        R fv[BT::NF ? K : 1][3], tv[BT::NT ? K : 1][3];
#pragma unroll
        for (int k = 0; k < K; ++k)
#pragma unroll
          for (int c = 0; c < 3; ++c) {
            fv[k][c] = R(0);
            tv[k][c] = R(0);
          }
        if (il < cnt) {
          const int64_t gj = Sy.b0 + s0 + il;
          double B;
          load_blob(p.r, gj, p.a, p.inva, X, Y, Z, B, DOM);
#pragma unroll
          for (int k = 0; k < K; ++k) {
            if constexpr (BT::NF) {
              const double* v = p.f + k * p.rhs_stride + 3 * gj;
              const double c = p.c1 * B;
              fv[k][0] = (R)(c * v[0]); fv[k][1] = (R)(c * v[1]); fv[k][2] = (R)(pz * c * v[2]);
            }
            if constexpr (BT::NT) {
              const double* v = p.t + k * p.rhs_stride + 3 * gj;
              const double c = p.c2 * B;
              tv[k][0] = (R)(c * v[0]); tv[k][1] = (R)(c * v[1]); tv[k][2] = (R)(pz * c * v[2]);
            }
          }
        }
        const int e0 = kDbl ? 128 * (il >> 6) + (il & 63) : il;
#pragma unroll
        for (int e = e0; e <= e0 + (kDbl ? 64 : 0); e += 64) {
          s_x[e] = X; s_y[e] = Y; s_z[e] = Z; s_zr[e] = (R)Z;
#pragma unroll
          for (int k = 0; k < K; ++k)
#pragma unroll
            for (int c = 0; c < 3; ++c) {
              if constexpr (BT::NF) s_f[k][c][e] = fv[k][c];
              if constexpr (BT::NT) s_t[k][c][e] = tv[k][c];
            }
        }
      }
      __syncthreads();
      const bool diag = S == T;
      // full off-diagonal tile pair: every lane's pair is taken, no masks.
      // Measured on MI355X with every kernel in one process, alternating:
      // the unmasked loop (8 fewer VALU per pair) makes the wall UF product
      // 17 % faster at 32768 blobs (fp32_blocked; 4 % in FP64) and UF + UT
      // 3 % faster; the two-output (grand) kernels keep the masked loop
      // only, as the second copy of their loop costs registers (K = 1:
      // 1 % slower; matrix form: 40 % slower).
      constexpr bool kUnmasked = DOM == kDomNoWall || DOM == kDomFreeSurface || (!kMat && OC == 3);
      const bool full = kUnmasked && !diag && cnt == kBlock && (T + 1) * kBlock <= Sy.n;
      for (int b = bb0; b < bb1 && 64 * b < cnt; ++b) {
        JT ja[K][OC];
#pragma unroll
        for (int k = 0; k < K; ++k)
#pragma unroll
          for (int c = 0; c < OC; ++c) ja[k][c] = JT(0);
        auto steps = [&](auto masked_c) {
        constexpr bool MASKED = decltype(masked_c)::value;
        for (int st = 0; st < 64; ++st) {
          const int jl = 64 * b + ((lane + st) & 63);   // the source, within the tile
          const int jr = kDbl ? 128 * b + lane + st : jl;   // its LDS entry
          const bool on = !MASKED || (valid && jl < cnt && (!diag || jl > il));
          const R zj = s_zr[jr];
          // matrix form (two waves per SIMD, too few to hide LDS latency):
          // the source's position, then its right-hand sides, read at the
          // top of the step in that order, so that the geometry waits for
          // the position only and the blocks' formation covers the rest
          // (2 % faster than reads where first used; FP32 pair terms only,
          // the FP64 kernels would lose a wave per SIMD to the registers)
          constexpr bool kEarly = kMat && !PER && sizeof(R) == 4;
          R fje[kEarly && BT::NF ? K : 1][3], tje[kEarly && BT::NT ? K : 1][3];
          double xje = 0.0, yje = 0.0, zje = 0.0;
          if constexpr (kEarly) {
            xje = s_x[jr]; yje = s_y[jr]; zje = s_z[jr];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int k = 0; k < K; ++k)
#pragma unroll
              for (int c = 0; c < 3; ++c) {
                if constexpr (BT::NF) fje[k][c] = s_f[k][c][jr];
                if constexpr (BT::NT) tje[k][c] = s_t[k][c][jr];
              }
            __builtin_amdgcn_sched_barrier(0);
          }
          // one image d = (dx, dy, dz) of the pair, applied on both sides; the
          // source-side sums move one lane per step (fused into the add; with
          // images, once per step before them)
          auto image = [&](auto rot_c, R dx, R dy, R dz, auto& sums) {
            mutual_apply<MASK, K, ACC, R, DOM, MASKED, decltype(rot_c)::value>(
                dx, dy, dz, zi, zj, on, fi, ti,
                [&](int k, int c) { return kEarly ? fje[kEarly ? k : 0][c] : s_f[k][c][jr]; },
                [&](int k, int c) { return kEarly ? tje[kEarly ? k : 0][c] : s_t[k][c][jr]; }, u, w, sums);
          };
          auto pair_apply = [&](R dx, R dy, R dz) { image(std::true_type{}, dx, dy, dz, ja); };
          if constexpr (kEarly) {
            if constexpr (sizeof(R) == 4)
              pair_apply((R)(Xi - xje), (R)(Yi - yje), (R)(Zi - zje));
            else
              pair_apply(Xi - xje, Yi - yje, Zi - zje);
          } else if constexpr (!PER) {
            if constexpr (sizeof(R) == 4)
              pair_apply((R)(Xi - s_x[jr]), (R)(Yi - s_y[jr]), (R)(Zi - s_z[jr]));
            else
              pair_apply(Xi - s_x[jr], Yi - s_y[jr], Zi - s_z[jr]);
          } else {
            ImageSum<ACC, R> ji[K][OC];
#pragma unroll
            for (int k = 0; k < K; ++k)
#pragma unroll
              for (int c = 0; c < OC; ++c) ji[k][c] = 0;
            each_image<R>(Xi - s_x[jr], Yi - s_y[jr], Zi - s_z[jr], p.periodic, p.L, p.iL,
                          [&](R dx, R dy, R dz, bool) { image(std::false_type{}, dx, dy, dz, ji); });
#pragma unroll
            for (int k = 0; k < K; ++k)
#pragma unroll
              for (int c = 0; c < OC; ++c) ja[k][c] = rol1(ja[k][c]) + (JT)ji[k][c];
          }
          if ((st & kFold) == kFold) {
            flush_all<K, ACC>(u, w);
            if constexpr (kFoldJ) {
              // lane l holds the sum of source (l + st) mod 64 of the block
              const int jw = (lane + st) & 63;
              // every read first, then the adds and writes: one LDS round
              // trip per fold (at the first fold of a block the reads return
              // stale values, a previous block's sums or uninitialised
              // memory, which the select drops)
              double prev[K][OC];
#pragma unroll
              for (int k = 0; k < K; ++k)
#pragma unroll
                for (int c = 0; c < OC; ++c) prev[k][c] = s_jd[wv][k][c][jw];
              const bool first = st <= kFold;
#pragma unroll
              for (int k = 0; k < K; ++k)
#pragma unroll
                for (int c = 0; c < OC; ++c) {
                  s_jd[wv][k][c][jw] = (first ? 0.0 : prev[k][c]) + (double)ja[k][c];
                  ja[k][c] = JT(0);
                }
            }
          }
        }
        };
        if constexpr (!kUnmasked) {
          steps(std::true_type{});
        } else {
          if (full) steps(std::false_type{}); else steps(std::true_type{});
        }
        if constexpr (!kFoldJ) {
          const int jw = (lane + 63) & 63;
#pragma unroll
          for (int k = 0; k < K; ++k)
#pragma unroll
            for (int c = 0; c < OC; ++c) s_jd[wv][k][c][jw] = (double)ja[k][c];
        }
        __syncthreads();  // every wave's sums of this block are in LDS
        if (il < 64 && 64 * b + il < cnt) {
          const int64_t slot = Sy.pj0 + tri_index(S, T);
#pragma unroll
          for (int k = 0; k < K; ++k) {
            double* P = p.part_j + ((slot * K + k) * kBlock + 64 * b + il) * OC;
#pragma unroll
            for (int c = 0; c < OC; ++c)
              P[c] = ((s_jd[0][k][c][il] + s_jd[1][k][c][il]) + s_jd[2][k][c][il]) + s_jd[3][k][c][il];
          }
        }
        __syncthreads();  // s_jd is free for the next block
      }
      flush_all<K, ACC>(u, w);
    }
    if (valid) {
      const int64_t slot = Sy.pi0 + local;
#pragma unroll
      for (int k = 0; k < K; ++k) {
        double* P = p.part_i + ((slot * K + k) * kBlock + il) * OC;
        int o = 0;
        if constexpr (BT::HU) {
          P[0] = u[k][0].get(); P[1] = u[k][1].get(); P[2] = u[k][2].get();
          o = 3;
        }
        if constexpr (BT::HW) {
          P[o] = w[k][0].get(); P[o + 1] = w[k][1].get(); P[o + 2] = w[k][2].get();
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// 4. reduce: fixed-order chunk sum + FP64 self term + damping.
// ---------------------------------------------------------------------------
struct ReduceParams {
  const double* r;
  const double* f;
  const double* t;
  double* vel;
  double* omg;
  const double* partial;
  const SysInfo* table;
  SysInfo single;
  int nsys;
  int mask;
  int K;
  int64_t ntot;
  int64_t rhs_stride, out_stride;  // doubles between RHS in f/t, in vel/omg
  double a, inva, c1, c2;
  int domain;
};

__device__ inline SysInfo find_sys_blob(const ReduceParams& p, int64_t gi)
{
  if (!p.table) return p.single;
  int lo = 0, hi = p.nsys - 1;
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if (p.table[mid].b0 <= gi) lo = mid; else hi = mid - 1;
  }
  return p.table[lo];
}

__global__ __launch_bounds__(256) void reduce_kernel(ReduceParams p)
{
  // one thread per (rhs k, blob gi, output component c in [0, OC))
  const bool HU = (p.mask & (kUF | kUT)) != 0;
  const bool HW = (p.mask & (kWF | kWT)) != 0;
  const int OC = 3 * ((HU ? 1 : 0) + (HW ? 1 : 0));
  const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t per_k = p.ntot * OC;
  if (tid >= per_k * p.K) return;
  const int k = (int)(tid / per_k);
  const int64_t rem = tid - (int64_t)k * per_k;
  const int64_t gi = rem / OC;
  const int c = (int)(rem - gi * OC);
  const SysInfo S = find_sys_blob(p, gi);
  const int64_t il = gi - S.b0;
  const double* P = p.partial + S.part0 + ((int64_t)k * S.n + il) * OC + c;
  const int64_t cstride = (int64_t)p.K * S.n * OC;
  double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
  int64_t ch = 0;
  for (; ch + 4 <= S.n_chunks; ch += 4) {
    s0 += P[(ch + 0) * cstride];
    s1 += P[(ch + 1) * cstride];
    s2 += P[(ch + 2) * cstride];
    s3 += P[(ch + 3) * cstride];
  }
  for (; ch < S.n_chunks; ++ch) s0 += P[ch * cstride];
  double sum = (s0 + s1) + (s2 + s3);

  finish_output(p.r, p.f, p.t, p.vel, p.omg, p.mask, k, gi, c, sum, p.rhs_stride, p.out_stride, p.a, p.inva,
                p.c1, p.c2, p.domain);
}

// Reduce of the symmetric path: for blob gi of tile X of its system, the
// target-side slots of X's items, then the source-side slots (X, T) for
// T = 0..X, each with two running sums, in that order.
struct MutReduceParams {
  const double* r;
  const double* f;
  const double* t;
  double* vel;
  double* omg;
  const double* part_i;
  const double* part_j;
  const MutSys* table;
  MutSys single;
  int nsys;
  int mask;
  int K;
  int64_t chunk_blocks;
  int64_t rhs_stride, out_stride;
  double a, inva, c1, c2;
  int domain;
  int periodic;             // bit d set when L_d > 0: add the self pair's outer images
  double L[3];              // periodic lengths / a
};

// Output o (component c of blob gi, RHS k) sums the target-side slots of the
// work items of its tile and the source-side slots (X, T), T <= X.  Eight
// groups of 32 threads share a workgroup's 32 outputs: group g takes slots
// g, g + 8, ... of both lists (consecutive threads read consecutive
// outputs of one slot), then group 0 adds the eight partial sums in order.
// The 32 outputs lie in one tile and right-hand side, which the workgroup's
// number gives: the search for the system and the divisions are scalar work
// (64 systems of 128 to 4096 blobs: 106 us with both per thread, in 64 bits, 76).
constexpr int kRedGroups = 8, kRedOut = 256 / kRedGroups;

// PER: pseudo-periodic calls, which add the self pair's outer images; the
// image loop takes 168 VGPRs, so calls without images run an instantiation
// without it (70 VGPRs: seven waves per SIMD instead of three for this
// latency-bound loop).
// BS: blobs per tile of the pair kernel (256, or the 64-blob blocks of
// rmw_wall_blocks.hip, whose work items are runs of chunk_blocks tiles).
template <bool PER, int BS>
__global__ __launch_bounds__(256) void mutual_reduce_kernel(MutReduceParams p)
{
  __shared__ double part[kRedGroups][kRedOut];
  const bool HU = (p.mask & (kUF | kUT)) != 0;
  const bool HW = (p.mask & (kWF | kWT)) != 0;
  const int OC = 3 * ((HU ? 1 : 0) + (HW ? 1 : 0));
  const int g = threadIdx.x / kRedOut, ol = threadIdx.x - g * kRedOut;
  constexpr int R3 = BS * 3 / kRedOut, R6 = BS * 6 / kRedOut;   // workgroups of one tile
  const int k = blockIdx.y;
  const int Xg = OC == 3 ? blockIdx.x / R3 : blockIdx.x / R6;   // the tile, among all systems'
  const int run = (int)blockIdx.x - Xg * (OC == 3 ? R3 : R6);
  MutSys Sy = p.single;
  if (p.table) {
    int lo = 0, hi = p.nsys - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (p.table[mid].t0 <= Xg) lo = mid; else hi = mid - 1;
    }
    Sy = p.table[lo];
  }
  const int64_t X = Xg - Sy.t0;
  const int e = run * kRedOut + ol;   // output within the tile
  const int l = OC == 3 ? e / 3 : e / 6, c = e - l * OC;
  const bool valid = X * BS + l < Sy.n;
  const int64_t gi = Sy.b0 + X * BS + l;
  double sum = 0.0;
  if (valid) {
    auto before = [&](int64_t x) {
      return BS == kBlock ? items_before_blocks(x, Sy.n_t, p.chunk_blocks) : items_before(x, Sy.n_t, p.chunk_blocks);
    };
    const int64_t it0 = before(X), it1 = before(X + 1);
    const int64_t step = (int64_t)p.K * BS * OC;
    const double* Pi = p.part_i + ((Sy.pi0 + it0) * p.K + k) * (BS * OC) + e;
    const double* Pj = p.part_j + ((Sy.pj0 + tri_index(X, 0)) * p.K + k) * (BS * OC) + e;
    // four loads in flight per thread (the loop is latency-bound: one
    // dependent load per slot took ~2x longer at 32768 blobs)
    auto strided_sum = [&](const double* P, int64_t cnt) {
      double a0 = 0.0, a1 = 0.0, a2 = 0.0, a3 = 0.0;
      int64_t m = g;
      for (; m + 3 * kRedGroups < cnt; m += 4 * kRedGroups) {
        a0 += P[m * step];
        a1 += P[(m + kRedGroups) * step];
        a2 += P[(m + 2 * kRedGroups) * step];
        a3 += P[(m + 3 * kRedGroups) * step];
      }
      for (; m < cnt; m += kRedGroups) a0 += P[m * step];
      return (a0 + a1) + (a2 + a3);
    };
    sum = strided_sum(Pi, it1 - it0) + strided_sum(Pj, X + 1);
  }
  part[g][ol] = sum;
  __syncthreads();
  if (g == 0 && valid) {
    double s = part[0][ol];
#pragma unroll
    for (int q = 1; q < kRedGroups; ++q) s += part[q][ol];
    finish_output(p.r, p.f, p.t, p.vel, p.omg, p.mask, k, gi, c, s, p.rhs_stride, p.out_stride, p.a, p.inva,
                  p.c1, p.c2, p.domain, PER ? p.periodic : 0, p.L[0], p.L[1], p.L[2]);
  }
}

// ---------------------------------------------------------------------------
// 5. optional check of the outputs (RMW_FLAG_CHECK_FINITE).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void copy_rows_kernel(const double* __restrict__ src, int64_t src_stride,
                                                        double* __restrict__ dst, int64_t dst_stride, int64_t len)
{
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < len) dst[blockIdx.y * dst_stride + i] = src[blockIdx.y * src_stride + i];
}

void launch_copy_rows(const double* src, int64_t src_stride, double* dst, int64_t dst_stride, int64_t len, int K,
                      hipStream_t st)
{
  for (int k = 0; k < K; k += 65535)
    hipLaunchKernelGGL(copy_rows_kernel, dim3((unsigned)((len + 255) / 256), std::min(K - k, 65535)), dim3(256), 0, st,
                       src + k * src_stride, src_stride, dst + k * dst_stride, dst_stride, len);
  RMW_CHECK_HIP(hipGetLastError());
}

__global__ void zero_count_kernel(unsigned int* count)
{
  if (threadIdx.x == 0) count[0] = 0u;
}

// count += number of inf / NaN entries among k rows of len doubles, rows
// `stride` apart.
__global__ __launch_bounds__(256) void count_nonfinite_kernel(const double* __restrict__ x, int64_t k, int64_t len,
                                                              int64_t stride, unsigned int* count)
{
  unsigned int bad = 0;
  const int64_t total = k * len;
  for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
       idx += (int64_t)gridDim.x * blockDim.x) {
    const int64_t row = idx / len;
    const double v = x[row * stride + (idx - row * len)];
    bad += isfinite(v) ? 0u : 1u;
  }
  if (bad) atomicAdd(count, bad);
}

// ---------------------------------------------------------------------------
// Host side: plan, workspace layout, dispatch.
// ---------------------------------------------------------------------------
// Vector with room for one element inside the object: the plan of a
// single suspension (every call but the ragged ones) uses no heap memory.
template <typename T>
class SmallVec {
 public:
  void push_back(const T& v)
  {
    if (n_ == 0 && heap_.empty()) {
      one_ = v;
    } else {
      if (heap_.empty()) heap_.push_back(one_);
      heap_.push_back(v);
    }
    ++n_;
  }
  size_t size() const { return n_; }
  bool empty() const { return n_ == 0; }
  void clear()
  {
    n_ = 0;
    heap_.clear();
  }
  const T* data() const { return heap_.empty() ? &one_ : heap_.data(); }
  const T& operator[](size_t i) const { return data()[i]; }

 private:
  T one_{};
  std::vector<T> heap_;
  size_t n_ = 0;
};

// Kernels a plan runs: the ordered kernel (source chunks, two launches), the
// symmetric kernel on 256-blob tiles or on 64-blob blocks, or the direct
// kernel (one launch).
enum : int { kOrderedPath, kTilesPath, kBlocksPath, kDirectPath };

struct Plan {
  int domain = kDomWall;
  int path = kOrderedPath;
  int mask = 0, prec = 0, kmax = 1;
  int slots = 0;             // resident pair-kernel workgroups on the device
  int64_t ntot = 0;
  SmallVec<SysInfo> sys;     // non-empty systems only
  int64_t total_items = 0;
  size_t partial_doubles = 0;
  size_t off_partial = 0, off_table = 0, total = 0;
  // symmetric paths
  bool over_cap = false;     // symmetric by its size, ordered because no layout fits
  int kmax_mut = 1;
  int64_t mut_items = 0, mut_tiles = 0, chunk_blocks = 4;   // symmetric work item: chunk_blocks 64-source blocks
  SmallVec<MutSys> msys;     // non-empty systems only
  size_t off_pi = 0, off_pj = 0, off_mtable = 0;
  // direct path
  int kmax_direct = 1;
  SmallVec<DirectSys> dsys;  // non-empty systems only
  int64_t direct_wgs = 0;
  size_t off_dtable = 0;
  // outputs of a product in place: all right-hand sides of the call
  size_t off_stage = 0, stage_bytes = 0;
  // RMW_FLAG_CHECK_FINITE: a counter of non-finite outputs after the rest
  bool check_finite = false;
  size_t off_status = 0;
};

static bool valid_mask(int mask) { return mask > 0 && mask < 16; }

// Right-hand sides per pair-kernel pass: 4, 2 or 1, at most the tuned cap.
static int group_k(int k, int cap)
{
  const int g = k >= 4 ? 4 : (k >= 2 ? 2 : 1);
  return cap > 0 && cap < g ? (cap >= 2 ? 2 : 1) : g;
}

static int rhs_cap(const rmw_tuning* tuning) { return tuning ? tuning->rhs_group : 0; }

constexpr int kChunkQuantum = 64;  // chunk lengths are multiples of this

template <int MASK, int K>
static const void* pair_ptr(int prec)
{
  if (prec == RMW_PREC_F32_F64ACC) return reinterpret_cast<const void*>(&pair_kernel_f32<MASK, K, RMW_PREC_F32_F64ACC>);
  if (prec == RMW_PREC_F32_BLOCKED) return reinterpret_cast<const void*>(&pair_kernel_f32<MASK, K, RMW_PREC_F32_BLOCKED>);
  if (prec == RMW_PREC_F32_KAHAN) return reinterpret_cast<const void*>(&pair_kernel_f32<MASK, K, RMW_PREC_F32_KAHAN>);
  return reinterpret_cast<const void*>(&pair_kernel_f64<MASK, K>);
}

template <int MASK>
static const void* pair_ptr_k(int prec, int K)
{
  return K == 4 ? pair_ptr<MASK, 4>(prec) : (K == 2 ? pair_ptr<MASK, 2>(prec) : pair_ptr<MASK, 1>(prec));
}

static const void* pair_kernel_ptr(int mask, int prec, int K)
{
  switch (mask) {
    case 1: return pair_ptr_k<1>(prec, K);
    case 2: return pair_ptr_k<2>(prec, K);
    case 3: return pair_ptr_k<3>(prec, K);
    case 4: return pair_ptr_k<4>(prec, K);
    case 5: return pair_ptr_k<5>(prec, K);
    case 8: return pair_ptr_k<8>(prec, K);
    case 10: return pair_ptr_k<10>(prec, K);
    case 12: return pair_ptr_k<12>(prec, K);
    default: return pair_ptr_k<15>(prec, K);
  }
}

// Workgroups of the (mask, prec, K) pair kernel resident on the whole
// device at once (register and LDS limited), cached per device.
static int resident_slots(int mask, int prec, int K)
{
  // fixed table (no heap use on the launch path): one entry per
  // (device, mask, prec, K) seen, first come first kept
  static std::mutex mu;
  static std::pair<int64_t, int> cache[256];
  static int used = 0;
  const DeviceProps& dp = device_props();
  const int64_t key = ((((int64_t)dp.device * 16 + mask) * 8 + prec) * 8) + K;
  {
    std::lock_guard<std::mutex> lk(mu);
    for (int i = 0; i < used; ++i)
      if (cache[i].first == key) return cache[i].second;
  }
  int per_cu = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, pair_kernel_ptr(mask, prec, K), kBlock, 0) !=
          hipSuccess ||
      per_cu < 1)
    per_cu = 1;
  const int slots = per_cu * std::max(dp.cu_count, 1);
  std::lock_guard<std::mutex> lk(mu);
  if (used < 256) cache[used++] = {key, slots};
  return slots;
}

// Built-in chunk length: ~16 work items per CU over the whole batch (small
// items keep the workgroups of a CU out of step and balance the persistent
// loop of ragged batches), at least one LDS tile.  The autotuner refines it.
static int64_t default_chunk(double pairs, int cu_count)
{
  const double c = pairs / (16.0 * std::max(cu_count, 1) * kBlock);
  return std::max<int64_t>(kBlock, (int64_t)std::ceil(c / kChunkQuantum) * kChunkQuantum);
}

// Blocks with a symmetric kernel: the UF block alone, UF + UT, the single UT,
// WF and WT blocks (UT_ji = WF_ij^T, WT_ji = WT_ij^T: a pair's source side
// of one of them is the transposed other) and all four, as far as the
// boundary serves them (the free surface: UF only; in plane: UF, UT, UF +
// UT); several right-hand sides per pass for UF and all four blocks above
// the wall, one otherwise.
static bool symmetric_mask(int mask, int domain)
{
  const bool single_rot = mask == kUT || mask == kWF || mask == kWT;
  return mask == kUF || ((mask == (kUF | kUT) || single_rot) && domain != kDomFreeSurface) ||
         (mask == (kUF | kUT | kWF | kWT) && (domain == kDomWall || domain == kDomNoWall));
}

// Ordered pairs up to which one direct launch is taken: the symmetric
// kernel on blocks evaluates half the pairs but takes two launches.  Measured
// (direct against blocks, us per product): UF fp32_blocked 6.5 / 11.4 at 1024
// blobs, 14.3 / 16.9 at 2048, 26.4 / 23.8 at 3000; FP64 17.9 / 20.8 and 34.3 /
// 31.4 at 2048 and 3000; all four blocks 26.1 / 28.0 and 50.0 / 40.2; UF + UT
// with nine images 39 / 59 at 1024, 99.6 / 96.9 at 2048.  Batches, whose
// workgroups are more than fit at once, up to a quarter of that, counting
// whole passes over 256 sources (all four blocks: 64 systems of 16 to 100
// blobs 19.7 / 24.9, 32 of 203 to 381 blobs 42 / 31).
constexpr double kDirectPairs = 2304.0 * 2304.0;

// Mean suspension size (weighted by blobs) up to which the symmetric kernel
// works on 64-blob blocks instead of 256-blob tiles.  Measured (blocks
// against tiles with 64-source items, us): UF fp32_blocked 36 / 39 at 4200,
// 55.2 / 54.2 at 6000, 133 / 129 at 10752; FP64 45 / 52, 77 / 81, 212 / 217;
// all four blocks 59 / 71, 105 / 108, 279 / 281; four right-hand sides of
// them 150 / 169 at 4200, 463 / 451 at 8192; UF + UT with images 470 / 548 at
// 6151, 753 / 819 at 8192.
static double block_kernel_blobs(int mask, int prec, int K, bool periodic)
{
  const bool light = K > 1 || (mask == kUF && prec != RMW_PREC_F64 && !periodic);
  return light ? 5632.0 : 9216.0;
}

// Non-empty systems of a direct launch with tt targets per workgroup.
static SmallVec<DirectSys> direct_table(const int64_t* offsets, int nsys, int tt, int64_t& wgs)
{
  SmallVec<DirectSys> table;
  wgs = 0;
  for (int s = 0; s < nsys; ++s) {
    const int64_t n = offsets[s + 1] - offsets[s];
    if (n == 0) continue;
    table.push_back(DirectSys{offsets[s], n, wgs});
    wgs += (n + tt - 1) / tt;
  }
  return table;
}

// offsets: host array of nsys + 1 blob offsets (offsets[0] = 0).  periodic:
// the call has pseudo-periodic images (the symmetric wall kernels then take
// one right-hand side per pass, so their partial sums are sized for one).
// stage: room for the outputs of a product in place.  cap: bytes that the
// partial sums of an automatically chosen symmetric layout may take.
static Plan make_plan(int mask, int prec, const int64_t* offsets, int nsys, int k,
                      const rmw_tuning* tuning, bool ragged, int domain = kDomWall, bool periodic = false,
                      bool stage = true, size_t cap = kMutAutoBytes)
{
  RMW_REQUIRE(valid_mask(mask), "mask must be a non-empty subset of UF|UT|WF|WT");
  RMW_REQUIRE(domain >= kDomWall && domain <= kDomFreeSurface, "unknown domain");
  RMW_REQUIRE(domain != kDomInPlane || (mask & ~(kUF | kUT)) == 0,
              "the in-plane mobility has the UF and UT blocks only");
  RMW_REQUIRE(domain != kDomFreeSurface || mask == kUF, "the free-surface mobility has the UF block only");
  RMW_REQUIRE(prec == RMW_PREC_F32_F64ACC || prec == RMW_PREC_F32_KAHAN || prec == RMW_PREC_F64 ||
                  prec == RMW_PREC_F32_BLOCKED,
              "unknown precision mode");
  RMW_REQUIRE(k >= 1, "k must be >= 1");
  Plan pl;
  pl.mask = mask;
  pl.prec = prec;
  pl.domain = domain;
  RMW_REQUIRE(!tuning || tuning->rhs_group == 0 || tuning->rhs_group == 1 || tuning->rhs_group == 2 ||
                  tuning->rhs_group == 4,
              "rhs_group must be 0, 1, 2 or 4");
  pl.kmax = group_k(k, domain == kDomWall ? rhs_cap(tuning) : 1);
  RMW_REQUIRE(offsets != nullptr && nsys >= 1 && offsets[0] == 0, "offsets must start at 0");
  for (int s = 0; s < nsys; ++s) RMW_REQUIRE(offsets[s + 1] >= offsets[s], "offsets must be non-decreasing");
  pl.ntot = offsets[nsys];

  double pairs = 0.0;
  int64_t nmax = 0;
  for (int s = 0; s < nsys; ++s) {
    double n = (double)(offsets[s + 1] - offsets[s]);
    pairs += n * n;
    nmax = std::max<int64_t>(nmax, offsets[s + 1] - offsets[s]);
  }
  pl.slots = resident_slots(mask, prec, pl.kmax);
  int64_t chunk = tuning && tuning->chunk_len > 0 ? tuning->chunk_len : 0;
  if (chunk <= 0) chunk = default_chunk(pairs, device_props().cu_count);
  chunk = std::max<int64_t>(kChunkQuantum, (chunk + kChunkQuantum - 1) / kChunkQuantum * kChunkQuantum);
  if (nmax > 0) chunk = std::min<int64_t>(chunk, (nmax + kChunkQuantum - 1) / kChunkQuantum * kChunkQuantum);

  const bool HU = (mask & (kUF | kUT)) != 0, HW = (mask & (kWF | kWT)) != 0;
  const int OC = 3 * ((HU ? 1 : 0) + (HW ? 1 : 0));
  int64_t item = 0, part = 0;
  for (int s = 0; s < nsys; ++s) {
    SysInfo S;
    S.b0 = offsets[s];
    S.n = offsets[s + 1] - offsets[s];
    if (S.n == 0) continue;
    S.n_tt = (S.n + kBlock - 1) / kBlock;
    S.chunk_len = chunk;
    S.n_chunks = (S.n + chunk - 1) / chunk;
    S.item0 = item;
    S.part0 = part;
    item += S.n_tt * S.n_chunks;
    part += S.n_chunks * (int64_t)pl.kmax * S.n * OC;
    pl.sys.push_back(S);
  }
  pl.total_items = item;
  pl.partial_doubles = (size_t)part;

  // The path.  A tuning that names a launch shape (chunk_len, max_wgs or
  // symmetric) gets the ordered or the tile kernel it was made for; the
  // built-in choice goes by the number of ordered pairs.
  const bool shaped = tuning && (tuning->chunk_len > 0 || tuning->max_wgs > 0 || tuning->symmetric != 0);
  const int sym = tuning ? tuning->symmetric : 0;
  const bool sym_mask = symmetric_mask(mask, domain);
  RMW_REQUIRE(!(sym > 0 && !(sym_mask && pl.ntot > 0)),
              "symmetric evaluation needs the UF block alone, UF + UT, one of UT, WF, WT, or all four blocks");
  const bool sym_ok = sym_mask && pl.ntot > 0 && (!periodic || domain == kDomWall);
  int64_t tile_pairs = 0, block_pairs = 0;
  double direct_work = 0.0;   // pairs, with the idle threads of a system's last 256 sources
  for (int s = 0; s < nsys; ++s) {
    const double n = (double)(offsets[s + 1] - offsets[s]);
    direct_work += n * (nsys > 1 ? std::ceil(n / kBlock) * kBlock : n);
    const int64_t nt = (offsets[s + 1] - offsets[s] + kBlock - 1) / kBlock;
    const int64_t nb = (offsets[s + 1] - offsets[s] + 63) / 64;
    tile_pairs += nt * (nt + 1) / 2;
    block_pairs += nb * (nb + 1) / 2;
  }
  const int cu = std::max(device_props().cu_count, 1);
  const int kgroup = periodic || domain != kDomWall || (mask != kUF && mask != 15) ? 1 : group_k(k, 4);
  const bool tiles_ok = sym_ok && (sym > 0 || (sym == 0 && tile_pairs >= cu));
  if (!shaped && direct_work <= (nsys > 1 ? 0.25 : 1.0) * kDirectPairs)
    pl.path = kDirectPath;
  else if (!shaped && sym_ok && pairs <= block_kernel_blobs(mask, prec, kgroup, periodic) * (double)pl.ntot)
    pl.path = kBlocksPath;
  else if (tiles_ok)
    pl.path = kTilesPath;

  size_t o = 0;
  if (pl.path == kTilesPath || pl.path == kBlocksPath) {
    // up to 4 right-hand sides per pass (each pair's blocks formed once as
    // 3x3 matrices and applied to all of them), fewer when the tuning caps it
    const int rc = rhs_cap(tuning);
    const bool single_rot = mask == kUT || mask == kWF || mask == kWT;
    pl.kmax_mut = domain == kDomWall && mask != (kUF | kUT) && !single_rot && !periodic
                      ? group_k(k, rc > 0 ? std::min(rc, 4) : 4)
                      : 1;
    // Layouts in the order of their speed; the first whose partial sums fit is
    // taken, with all right-hand sides of a pass before two (the source-side
    // slots grow as N^2 and with the right-hand sides), and the ordered kernel
    // where nothing fits.  ms for four right-hand sides of all four blocks:
    // 96 systems of 4096 blobs, two per pass by blocks 12.9, four by tiles 10.0;
    // 192, ordered 35.9, tiles 20.6; one of 64000, 26.7 / 23.1 (two / four);
    // 90000, ordered 60.3, two per pass 53.4.  In the library's own array two
    // right-hand sides fit only in runs that keep few CUs busy: there the ordered
    // kernel comes next (10000 blobs: 0.80, two per pass 0.97).
    const bool fewer = rc <= 0 && cap >= kMutAutoBytes;
    struct Layout { bool blk; int64_t chunk; };
    Layout layouts[3];
    int count = 0;
    if (pl.path == kBlocksPath) {
      // runs of one source block while that leaves a CU fewer than 12 work
      // items, then two (fewer target-side sums: UF fp32_blocked 141.6 ->
      // 132.5 us at 10752 blobs), four for large batches; with images one
      // up to three times that (478 against 501 us at 6151 before the divisions
      // for the images went)
      const int64_t fine = (periodic ? 36 : 12) * (int64_t)cu;
      layouts[count++] = {true, block_pairs <= fine ? 1 : (block_pairs <= 144 * (int64_t)cu ? 2 : 4)};
    }
    if (tuning && tuning->chunk_len > 0) {
      // 64 or 128 sources: a quarter or half of a tile pair per work item
      // (finer work for suspensions of few tiles); else whole source tiles
      const int64_t blocks = (tuning->chunk_len + 63) / 64;
      layouts[count++] = {false, blocks <= 2 ? blocks : (blocks + 3) / 4 * 4};
    } else if (tiles_ok) {
      // quarter tiles while they balance the CUs better than they cost in
      // partial sums, then half and whole tiles (us at 64 / 128 / 256 sources:
      // UF fp32_blocked 129 / 139 / 152 at 10752 blobs, 618 / 575 / 589 at 24576,
      // 1777 / 1694 / 1676 at 43008; four right-hand sides of all four blocks
      // 882 / 866 / 967 at 12000, 6271 / 6089 / 6081 at 32768); runs of tiles
      // with a third of the target-side sums where those do not fit
      const int64_t quarter = (pl.kmax_mut > 1 ? 4 : 8) * (int64_t)cu + 64;
      layouts[count++] = {false, tile_pairs <= quarter ? 1
                                 : tile_pairs <= 36 * (int64_t)cu
                                     ? 2
                                     : 4 * std::max<int64_t>(1, tile_pairs / (48 * (int64_t)cu))};
      layouts[count++] = {false, 4 * std::max<int64_t>(1, tile_pairs / (16 * (int64_t)cu))};
    }
    bool fits = false;
    for (int q = 0; !fits; ++q) {
      if (q == count) {   // no layout: two right-hand sides per pass, or a required one beyond the limit
        if (fewer && pl.kmax_mut > 2) {
          pl.kmax_mut = 2;
          q = 0;
        } else {
          if (sym <= 0) break;
          fits = true;
          q = count - 1;
        }
      }
      const bool blk = layouts[q].blk;
      const int64_t bs = blk ? 64 : kBlock, chunk_blocks = layouts[q].chunk;
      int64_t item = 0, pj = 0, tiles = 0;
      pl.msys.clear();
      for (int s = 0; s < nsys; ++s) {
        MutSys M;
        M.b0 = offsets[s];
        M.n = offsets[s + 1] - offsets[s];
        if (M.n == 0) continue;
        M.n_t = (M.n + bs - 1) / bs;
        M.item0 = item;
        M.pi0 = item;
        M.pj0 = pj;
        M.t0 = tiles;
        tiles += M.n_t;
        item += blk ? items_before(M.n_t, M.n_t, chunk_blocks) : items_before_blocks(M.n_t, M.n_t, chunk_blocks);
        pj += M.n_t * (M.n_t + 1) / 2;
        pl.msys.push_back(M);
      }
      const size_t slot = (size_t)pl.kmax_mut * bs * OC * sizeof(double);
      o = 0;
      pl.off_pi = o; o = align_up(o + (size_t)item * slot);
      pl.off_pj = o; o = align_up(o + (size_t)pj * slot);
      if (pl.msys.size() > 1) { pl.off_mtable = o; o = align_up(o + pl.msys.size() * sizeof(MutSys)); }
      fits = fits || o <= cap;
      pl.path = blk ? kBlocksPath : kTilesPath;
      pl.chunk_blocks = chunk_blocks;
      pl.mut_items = item;
      pl.mut_tiles = tiles;
    }
    if (!fits) {
      pl.over_cap = true;
      pl.path = kOrderedPath;
      pl.msys.clear();
      o = 0;
    }
  }
  if (pl.path == kDirectPath) {
    pl.kmax_direct = group_k(k, std::min(direct_max_k(mask, domain), rhs_cap(tuning) > 0 ? rhs_cap(tuning) : 4));
    pl.dsys = direct_table(offsets, nsys, direct_targets(mask, pl.kmax_direct), pl.direct_wgs);
    if (pl.dsys.size() > 1) { pl.off_dtable = o; o = align_up(o + pl.dsys.size() * sizeof(DirectSys)); }
  }
  if (pl.path == kOrderedPath) {
    pl.off_partial = o; o = align_up(o + pl.partial_doubles * sizeof(double));
    if (ragged) { pl.off_table = o; o = align_up(o + pl.sys.size() * sizeof(SysInfo)); }
  }
  if (stage) {
    pl.off_stage = o;
    pl.stage_bytes = align_up((size_t)k * pl.ntot * OC * sizeof(double));
    o += pl.stage_bytes;
  }
  pl.total = o;
  pl.check_finite = tuning && (tuning->flags & RMW_FLAG_CHECK_FINITE) != 0;
  if (pl.check_finite) {
    pl.off_status = align_up(pl.total);
    pl.total = pl.off_status + RMW_STATUS_BYTES;
  }
  return pl;
}

// Pair-kernel launch for one (MASK, K) instantiation.
template <int MASK, int K>
static void launch_pair(int prec, const PairParams& pp, int grid, hipStream_t st)
{
  if (prec == RMW_PREC_F32_F64ACC)
    hipLaunchKernelGGL((pair_kernel_f32<MASK, K, RMW_PREC_F32_F64ACC>), dim3(grid), dim3(kBlock), 0, st, pp);
  else if (prec == RMW_PREC_F32_BLOCKED)
    hipLaunchKernelGGL((pair_kernel_f32<MASK, K, RMW_PREC_F32_BLOCKED>), dim3(grid), dim3(kBlock), 0, st, pp);
  else if (prec == RMW_PREC_F32_KAHAN)
    hipLaunchKernelGGL((pair_kernel_f32<MASK, K, RMW_PREC_F32_KAHAN>), dim3(grid), dim3(kBlock), 0, st, pp);
  else
    hipLaunchKernelGGL((pair_kernel_f64<MASK, K>), dim3(grid), dim3(kBlock), 0, st, pp);
}

template <int MASK>
static void launch_pair_k(int prec, int K, const PairParams& pp, int grid, hipStream_t st)
{
  if (K == 4) launch_pair<MASK, 4>(prec, pp, grid, st);
  else if (K == 2) launch_pair<MASK, 2>(prec, pp, grid, st);
  else launch_pair<MASK, 1>(prec, pp, grid, st);
}

// Pair kernels of the no-wall, in-plane and free-surface products (one
// right-hand side per pass).
template <int MASK, int DOM>
static void launch_pair_dom(int prec, const PairParams& pp, int grid, hipStream_t st)
{
  const dim3 g(grid), b(kBlock);
  if (prec == RMW_PREC_F32_F64ACC)
    hipLaunchKernelGGL((pair_kernel_f32<MASK, 1, RMW_PREC_F32_F64ACC, DOM>), g, b, 0, st, pp);
  else if (prec == RMW_PREC_F32_BLOCKED)
    hipLaunchKernelGGL((pair_kernel_f32<MASK, 1, RMW_PREC_F32_BLOCKED, DOM>), g, b, 0, st, pp);
  else if (prec == RMW_PREC_F32_KAHAN)
    hipLaunchKernelGGL((pair_kernel_f32<MASK, 1, RMW_PREC_F32_KAHAN, DOM>), g, b, 0, st, pp);
  else
    hipLaunchKernelGGL((pair_kernel_f64<MASK, 1, DOM>), g, b, 0, st, pp);
}

static void dispatch_pair_domain(int domain, int mask, int prec, const PairParams& pp, int grid, hipStream_t st)
{
  if (domain == kDomFreeSurface) return launch_pair_dom<kUF, kDomFreeSurface>(prec, pp, grid, st);
  if (domain == kDomInPlane) {
    switch (mask) {
      case 1: return launch_pair_dom<1, kDomInPlane>(prec, pp, grid, st);
      case 2: return launch_pair_dom<2, kDomInPlane>(prec, pp, grid, st);
      default: return launch_pair_dom<3, kDomInPlane>(prec, pp, grid, st);
    }
  }
  switch (mask) {
    case 1: return launch_pair_dom<1, kDomNoWall>(prec, pp, grid, st);
    case 2: return launch_pair_dom<2, kDomNoWall>(prec, pp, grid, st);
    case 3: return launch_pair_dom<3, kDomNoWall>(prec, pp, grid, st);
    case 4: return launch_pair_dom<4, kDomNoWall>(prec, pp, grid, st);
    case 5: return launch_pair_dom<5, kDomNoWall>(prec, pp, grid, st);
    case 8: return launch_pair_dom<8, kDomNoWall>(prec, pp, grid, st);
    case 10: return launch_pair_dom<10, kDomNoWall>(prec, pp, grid, st);
    case 12: return launch_pair_dom<12, kDomNoWall>(prec, pp, grid, st);
    default: return launch_pair_dom<15, kDomNoWall>(prec, pp, grid, st);
  }
}

static void dispatch_pair(int mask, int prec, int K, const PairParams& pp, int grid, hipStream_t st)
{
  switch (mask) {
    case 1: launch_pair_k<1>(prec, K, pp, grid, st); break;
    case 2: launch_pair_k<2>(prec, K, pp, grid, st); break;
    case 3: launch_pair_k<3>(prec, K, pp, grid, st); break;
    case 4: launch_pair_k<4>(prec, K, pp, grid, st); break;
    case 5: launch_pair_k<5>(prec, K, pp, grid, st); break;
    case 8: launch_pair_k<8>(prec, K, pp, grid, st); break;
    case 10: launch_pair_k<10>(prec, K, pp, grid, st); break;
    case 12: launch_pair_k<12>(prec, K, pp, grid, st); break;
    default: launch_pair_k<15>(prec, K, pp, grid, st); break;
  }
}

// Masks with their own instantiation; the rest are rejected.
static int kernel_mask(int mask)
{
  switch (mask) {
    case 1: case 2: case 3: case 4: case 5: case 8: case 10: case 12: case 15: return mask;
    default: return 0;
  }
}

// Pinned host staging ring for small stream-ordered uploads (the ragged
// work table).  A slot is reused only after the copy that last read it has
// completed, so callers may free their host data right after the call.
struct StageSlot {
  void* host = nullptr;
  size_t cap = 0;
  hipEvent_t done = nullptr;
  bool pending = false;
};
static std::mutex g_stage_mu;
static StageSlot g_stage[8];
static int g_stage_next = 0;

static void stage_upload(void* dst, const void* src, size_t bytes, hipStream_t st)
{
  if (bytes == 0) return;
  std::lock_guard<std::mutex> lk(g_stage_mu);
  StageSlot& s = g_stage[g_stage_next];
  g_stage_next = (g_stage_next + 1) % 8;
  if (s.pending) {
    RMW_CHECK_HIP(hipEventSynchronize(s.done));
    s.pending = false;
  }
  if (s.cap < bytes) {
    if (s.host) RMW_CHECK_HIP(hipHostFree(s.host));
    s.host = nullptr;
    size_t cap = align_up(bytes, 4096);
    RMW_CHECK_HIP(hipHostMalloc(&s.host, cap, hipHostMallocDefault));
    s.cap = cap;
  }
  if (!s.done) RMW_CHECK_HIP(hipEventCreateWithFlags(&s.done, hipEventDisableTiming));
  std::memcpy(s.host, src, bytes);
  RMW_CHECK_HIP(hipMemcpyAsync(dst, s.host, bytes, hipMemcpyHostToDevice, st));
  RMW_CHECK_HIP(hipEventRecord(s.done, st));
  s.pending = true;
}

void stage_upload_public(void* dst, const void* src, size_t bytes, hipStream_t st)
{
  stage_upload(dst, src, bytes, st);
}

static std::mutex g_prof_mu;
static bool g_prof_on = false;
static std::vector<ProfRec> g_prof;

template <int MASK, int DOM>
static void dispatch_mutual_dom(int prec, const MutParams& q, int grid, hipStream_t st)
{
  const dim3 g(grid), b(kBlock);
  if (prec == RMW_PREC_F32_BLOCKED)
    hipLaunchKernelGGL((mutual_kernel<MASK, 1, RMW_PREC_F32_BLOCKED, float, DOM>), g, b, 0, st, q);
  else if (prec == RMW_PREC_F32_F64ACC)
    hipLaunchKernelGGL((mutual_kernel<MASK, 1, RMW_PREC_F32_F64ACC, float, DOM>), g, b, 0, st, q);
  else if (prec == RMW_PREC_F32_KAHAN)
    hipLaunchKernelGGL((mutual_kernel<MASK, 1, RMW_PREC_F32_KAHAN, float, DOM>), g, b, 0, st, q);
  else
    hipLaunchKernelGGL((mutual_kernel<MASK, 1, RMW_PREC_F64, double, DOM>), g, b, 0, st, q);
}

template <int MASK>
static void dispatch_mutual_m(int prec, int K, const MutParams& q, int grid, hipStream_t st)
{
  const dim3 g(grid), b(kBlock);
  if (prec == RMW_PREC_F32_BLOCKED) {
    if (K == 4) hipLaunchKernelGGL((mutual_kernel<MASK, 4, RMW_PREC_F32_BLOCKED, float>), g, b, 0, st, q);
    else if (K == 2) hipLaunchKernelGGL((mutual_kernel<MASK, 2, RMW_PREC_F32_BLOCKED, float>), g, b, 0, st, q);
    else hipLaunchKernelGGL((mutual_kernel<MASK, 1, RMW_PREC_F32_BLOCKED, float>), g, b, 0, st, q);
  } else if (prec == RMW_PREC_F32_F64ACC) {
    if (K == 4) hipLaunchKernelGGL((mutual_kernel<MASK, 4, RMW_PREC_F32_F64ACC, float>), g, b, 0, st, q);
    else if (K == 2) hipLaunchKernelGGL((mutual_kernel<MASK, 2, RMW_PREC_F32_F64ACC, float>), g, b, 0, st, q);
    else hipLaunchKernelGGL((mutual_kernel<MASK, 1, RMW_PREC_F32_F64ACC, float>), g, b, 0, st, q);
  } else if (prec == RMW_PREC_F32_KAHAN) {
    if (K == 4) hipLaunchKernelGGL((mutual_kernel<MASK, 4, RMW_PREC_F32_KAHAN, float>), g, b, 0, st, q);
    else if (K == 2) hipLaunchKernelGGL((mutual_kernel<MASK, 2, RMW_PREC_F32_KAHAN, float>), g, b, 0, st, q);
    else hipLaunchKernelGGL((mutual_kernel<MASK, 1, RMW_PREC_F32_KAHAN, float>), g, b, 0, st, q);
  } else {
    if (K == 4) hipLaunchKernelGGL((mutual_kernel<MASK, 4, RMW_PREC_F64, double>), g, b, 0, st, q);
    else if (K == 2) hipLaunchKernelGGL((mutual_kernel<MASK, 2, RMW_PREC_F64, double>), g, b, 0, st, q);
    else hipLaunchKernelGGL((mutual_kernel<MASK, 1, RMW_PREC_F64, double>), g, b, 0, st, q);
  }
}

// Pseudo-periodic images (wall domain, one right-hand side per pass).
template <int MASK>
static void dispatch_mutual_per_m(int prec, const MutParams& q, int grid, hipStream_t st)
{
  const dim3 g(grid), b(kBlock);
  if (prec == RMW_PREC_F32_BLOCKED)
    hipLaunchKernelGGL((mutual_kernel<MASK, 1, RMW_PREC_F32_BLOCKED, float, kDomWall, true>), g, b, 0, st, q);
  else if (prec == RMW_PREC_F32_F64ACC)
    hipLaunchKernelGGL((mutual_kernel<MASK, 1, RMW_PREC_F32_F64ACC, float, kDomWall, true>), g, b, 0, st, q);
  else if (prec == RMW_PREC_F32_KAHAN)
    hipLaunchKernelGGL((mutual_kernel<MASK, 1, RMW_PREC_F32_KAHAN, float, kDomWall, true>), g, b, 0, st, q);
  else
    hipLaunchKernelGGL((mutual_kernel<MASK, 1, RMW_PREC_F64, double, kDomWall, true>), g, b, 0, st, q);
}

static void dispatch_mutual_periodic(int mask, int prec, const MutParams& q, int grid, hipStream_t st)
{
  if (mask == kUF) dispatch_mutual_per_m<kUF>(prec, q, grid, st);
  else if (mask == (kUF | kUT)) dispatch_mutual_per_m<kUF | kUT>(prec, q, grid, st);
  else if (mask == kUT) dispatch_mutual_per_m<kUT>(prec, q, grid, st);
  else if (mask == kWF) dispatch_mutual_per_m<kWF>(prec, q, grid, st);
  else if (mask == kWT) dispatch_mutual_per_m<kWT>(prec, q, grid, st);
  else dispatch_mutual_per_m<kUF | kUT | kWF | kWT>(prec, q, grid, st);
}

static void dispatch_mutual(int domain, int mask, int prec, int K, const MutParams& q, int grid, hipStream_t st)
{
  if (domain == kDomNoWall) {
    if (mask == kUF) dispatch_mutual_dom<kUF, kDomNoWall>(prec, q, grid, st);
    else if (mask == (kUF | kUT)) dispatch_mutual_dom<kUF | kUT, kDomNoWall>(prec, q, grid, st);
    else if (mask == kUT) dispatch_mutual_dom<kUT, kDomNoWall>(prec, q, grid, st);
    else if (mask == kWF) dispatch_mutual_dom<kWF, kDomNoWall>(prec, q, grid, st);
    else if (mask == kWT) dispatch_mutual_dom<kWT, kDomNoWall>(prec, q, grid, st);
    else dispatch_mutual_dom<kUF | kUT | kWF | kWT, kDomNoWall>(prec, q, grid, st);
  } else if (domain == kDomInPlane) {
    if (mask == kUF) dispatch_mutual_dom<kUF, kDomInPlane>(prec, q, grid, st);
    else if (mask == (kUF | kUT)) dispatch_mutual_dom<kUF | kUT, kDomInPlane>(prec, q, grid, st);
    else dispatch_mutual_dom<kUT, kDomInPlane>(prec, q, grid, st);
  } else if (domain == kDomFreeSurface) {
    dispatch_mutual_dom<kUF, kDomFreeSurface>(prec, q, grid, st);
  } else if (mask == kUF) {
    dispatch_mutual_m<kUF>(prec, K, q, grid, st);
  } else if (mask == (kUF | kUT)) {
    // u = UF f + UT t: target side UF, UT; source side UF^T f_i + WF^T t_i
    dispatch_mutual_dom<kUF | kUT, kDomWall>(prec, q, grid, st);
  } else if (mask == kUT) {
    // u = UT t: target side UT t_j, source side WF^T t_i
    dispatch_mutual_dom<kUT, kDomWall>(prec, q, grid, st);
  } else if (mask == kWF) {
    // w = WF f: target side WF f_j, source side UT^T f_i
    dispatch_mutual_dom<kWF, kDomWall>(prec, q, grid, st);
  } else if (mask == kWT) {
    dispatch_mutual_dom<kWT, kDomWall>(prec, q, grid, st);
  } else {
    dispatch_mutual_m<kUF | kUT | kWF | kWT>(prec, K, q, grid, st);
  }
}

// Set while the calling thread runs rmw_wall_rpy_apply_noalloc: its
// launches take no timing records (each record creates two HIP events).
static thread_local bool tl_no_records = false;

// Pair-kernel timing records (rmw_profile_*).
void prof_begin(ProfRec& rec, bool& on, hipStream_t st, int kind)
{
  rec.kind = kind;
  {
    std::lock_guard<std::mutex> lk(g_prof_mu);
    on = g_prof_on && !tl_no_records;
  }
  if (on) {
    RMW_CHECK_HIP(hipEventCreate(&rec.a));
    RMW_CHECK_HIP(hipEventCreate(&rec.b));
    RMW_CHECK_HIP(hipEventRecord(rec.a, st));
  }
}

void prof_end(const ProfRec& rec, bool on, hipStream_t st)
{
  if (on) {
    RMW_CHECK_HIP(hipEventRecord(rec.b, st));
    std::lock_guard<std::mutex> lk(g_prof_mu);
    g_prof.push_back(rec);
  }
}

static void run_mutual(const Plan& pl, const double* r, const double* f, const double* t, double* vel,
                       double* omg, int k, int64_t stride, int64_t out_stride, double a, double inva, double c1,
                       double c2, const rmw_tuning* tuning, char* base, hipStream_t st, int periodic,
                       const double* Lp)
{
  const bool HU = (pl.mask & (kUF | kUT)) != 0, HW = (pl.mask & (kWF | kWT)) != 0;
  const bool NF = (pl.mask & (kUF | kWF)) != 0, NT = (pl.mask & (kUT | kWT)) != 0;
  MutSys* dtable = nullptr;
  if (pl.msys.size() > 1) {
    dtable = (MutSys*)(base + pl.off_mtable);
    stage_upload(dtable, pl.msys.data(), pl.msys.size() * sizeof(MutSys), st);
  }
  int grid = (int)std::min<int64_t>(pl.mut_items, (int64_t)INT32_MAX);
  if (tuning && tuning->max_wgs > 0) grid = std::min(grid, tuning->max_wgs);
  const int kmax = pl.kmax_mut;
  for (int k0 = 0, K = group_k(k, kmax); k0 < k; k0 += K) {
    K = group_k(k - k0, kmax);
    MutParams q{};
    q.r = r;
    q.f = NF ? f + (size_t)k0 * stride : nullptr;
    q.t = NT ? t + (size_t)k0 * stride : nullptr;
    q.rhs_stride = stride;
    q.a = a; q.inva = inva; q.c1 = c1; q.c2 = c2;
    q.part_i = (double*)(base + pl.off_pi);
    q.part_j = (double*)(base + pl.off_pj);
    q.table = dtable;
    q.single = pl.msys[0];
    q.nsys = (int)pl.msys.size();
    q.n_items = pl.mut_items;
    q.chunk_blocks = pl.chunk_blocks;
    q.periodic = periodic;
    for (int d = 0; d < 3; ++d) { q.L[d] = Lp[d]; q.iL[d] = Lp[d] > 0.0 ? 1.0 / Lp[d] : 0.0; }
    ProfRec rec{};
    bool prof = false;
    prof_begin(rec, prof, st);
    if (pl.path == kBlocksPath) launch_blocks(pl.domain, pl.mask, pl.prec, K, q, grid, st);
    else if (periodic) dispatch_mutual_periodic(pl.mask, pl.prec, q, grid, st);
    else dispatch_mutual(pl.domain, pl.mask, pl.prec, K, q, grid, st);
    RMW_CHECK_HIP(hipGetLastError());
    prof_end(rec, prof, st);

    MutReduceParams rp{};
    rp.r = r;
    rp.f = q.f; rp.t = q.t;
    rp.vel = HU ? vel + (size_t)k0 * out_stride : nullptr;
    rp.omg = HW ? omg + (size_t)k0 * out_stride : nullptr;
    rp.part_i = q.part_i;
    rp.part_j = q.part_j;
    rp.table = dtable;
    rp.single = q.single;
    rp.nsys = q.nsys;
    rp.mask = pl.mask;
    rp.K = K;
    rp.chunk_blocks = pl.chunk_blocks;
    rp.rhs_stride = stride;
    rp.out_stride = out_stride;
    rp.a = a; rp.inva = inva; rp.c1 = c1; rp.c2 = c2;
    rp.domain = pl.domain;
    rp.periodic = periodic;
    for (int d = 0; d < 3; ++d) rp.L[d] = Lp[d];
    const int OC = 3 * ((HU ? 1 : 0) + (HW ? 1 : 0));
    const int64_t tile_out = (pl.path == kBlocksPath ? 64 : kBlock) * OC;
    const dim3 rgrid((unsigned)(pl.mut_tiles * (tile_out / kRedOut)), K);
    const dim3 rb(256);
    if (pl.path == kBlocksPath) {
      if (periodic) hipLaunchKernelGGL((mutual_reduce_kernel<true, 64>), rgrid, rb, 0, st, rp);
      else hipLaunchKernelGGL((mutual_reduce_kernel<false, 64>), rgrid, rb, 0, st, rp);
    } else {
      if (periodic) hipLaunchKernelGGL((mutual_reduce_kernel<true, kBlock>), rgrid, rb, 0, st, rp);
      else hipLaunchKernelGGL((mutual_reduce_kernel<false, kBlock>), rgrid, rb, 0, st, rp);
    }
    RMW_CHECK_HIP(hipGetLastError());
  }
}

static void run_direct(const Plan& pl, const double* r, const double* f, const double* t, double* vel, double* omg,
                       int k, int64_t stride, int64_t out_stride, double a, double inva, double c1, double c2,
                       char* base, hipStream_t st, int periodic, const double* Lp)
{
  SmallVec<DirectSys> table = pl.dsys;
  int64_t wgs = pl.direct_wgs;
  DirectSys* dtable = nullptr;
  auto upload = [&] {
    if (table.size() > 1) {
      dtable = (DirectSys*)(base + pl.off_dtable);
      stage_upload(dtable, table.data(), table.size() * sizeof(DirectSys), st);
    }
  };
  upload();
  int tt = direct_targets(pl.mask, pl.kmax_direct);
  for (int k0 = 0, K = pl.kmax_direct; k0 < k; k0 += K) {
    K = group_k(k - k0, pl.kmax_direct);
    if (direct_targets(pl.mask, K) != tt) {   // a smaller last group: more targets per workgroup
      tt = direct_targets(pl.mask, K);
      wgs = 0;
      SmallVec<DirectSys> t2;
      for (size_t s = 0; s < table.size(); ++s) {
        t2.push_back(DirectSys{table[s].b0, table[s].n, wgs});
        wgs += (table[s].n + tt - 1) / tt;
      }
      table = t2;
      upload();
    }
    DirectParams q{};
    q.r = r;
    q.f = f ? f + (size_t)k0 * stride : nullptr;
    q.t = t ? t + (size_t)k0 * stride : nullptr;
    q.vel = vel ? vel + (size_t)k0 * out_stride : nullptr;
    q.omg = omg ? omg + (size_t)k0 * out_stride : nullptr;
    q.rhs_stride = stride;
    q.out_stride = out_stride;
    q.a = a; q.inva = inva; q.c1 = c1; q.c2 = c2;
    q.table = dtable;
    q.single = table[0];
    q.nsys = (int)table.size();
    q.periodic = periodic;
    for (int d = 0; d < 3; ++d) { q.L[d] = Lp[d]; q.iL[d] = Lp[d] > 0.0 ? 1.0 / Lp[d] : 0.0; }
    ProfRec rec{};
    bool prof = false;
    prof_begin(rec, prof, st);
    launch_direct(pl.domain, pl.mask, pl.prec, K, q, wgs, st);
    RMW_CHECK_HIP(hipGetLastError());
    prof_end(rec, prof, st);
  }
}

static void run_ordered(const Plan& pl, const double* r, const double* f, const double* t, double* vel, double* omg,
                        int k, int64_t stride, int64_t out_stride, double a, double inva, double c1, double c2,
                        const rmw_tuning* tuning, char* base, hipStream_t st, int periodic, const double* Lp,
                        bool ragged)
{
  const bool HU = (pl.mask & (kUF | kUT)) != 0, HW = (pl.mask & (kWF | kWT)) != 0;
  const bool NF = (pl.mask & (kUF | kWF)) != 0, NT = (pl.mask & (kUT | kWT)) != 0;
  SysInfo* dtable = nullptr;
  if (ragged) {
    dtable = (SysInfo*)(base + pl.off_table);
    stage_upload(dtable, pl.sys.data(), pl.sys.size() * sizeof(SysInfo), st);
  }

  int grid = (int)std::min<int64_t>(pl.total_items, (int64_t)INT32_MAX);
  if (ragged || (tuning && tuning->max_wgs > 0)) {
    const int cap = tuning && tuning->max_wgs > 0 ? tuning->max_wgs : std::max(pl.slots, 1);
    grid = (int)std::min<int64_t>(grid, cap);
  }

  const int kcap = pl.domain == kDomWall ? rhs_cap(tuning) : 1;
  for (int k0 = 0, K = group_k(k, kcap); k0 < k; k0 += K) {
    K = group_k(k - k0, kcap);
    PairParams q{};
    q.r = r;
    q.f = NF ? f + (size_t)k0 * stride : nullptr;
    q.t = NT ? t + (size_t)k0 * stride : nullptr;
    q.rhs_stride = stride;
    q.a = a; q.inva = inva; q.c1 = c1; q.c2 = c2;
    q.partial = (double*)(base + pl.off_partial);
    q.table = dtable;
    q.single = pl.sys.empty() ? SysInfo{} : pl.sys[0];
    q.nsys = (int)pl.sys.size();
    q.ntot = pl.ntot;
    q.total_items = pl.total_items;
    q.periodic = periodic;
    for (int d = 0; d < 3; ++d) { q.L[d] = Lp[d]; q.iL[d] = Lp[d] > 0.0 ? 1.0 / Lp[d] : 0.0; }
    q.domain = pl.domain;
    // The partial layout was planned for kmax RHS; a smaller trailing group
    // reuses it with its own K (items only touch their own slots).
    ProfRec rec{};
    bool prof = false;
    prof_begin(rec, prof, st);
    if (pl.domain == kDomWall) dispatch_pair(pl.mask, pl.prec, K, q, grid, st);
    else dispatch_pair_domain(pl.domain, pl.mask, pl.prec, q, grid, st);
    RMW_CHECK_HIP(hipGetLastError());
    prof_end(rec, prof, st);

    ReduceParams rp{};
    rp.r = r;
    rp.f = q.f; rp.t = q.t;
    rp.vel = HU ? vel + (size_t)k0 * out_stride : nullptr;
    rp.omg = HW ? omg + (size_t)k0 * out_stride : nullptr;
    rp.partial = q.partial;
    rp.table = dtable;
    rp.single = q.single;
    rp.nsys = q.nsys;
    rp.mask = pl.mask;
    rp.K = K;
    rp.ntot = pl.ntot;
    rp.rhs_stride = stride;
    rp.out_stride = out_stride;
    rp.a = a; rp.inva = inva; rp.c1 = c1; rp.c2 = c2;
    rp.domain = pl.domain;
    const int OCr = 3 * ((HU ? 1 : 0) + (HW ? 1 : 0));
    const int64_t nthreads = pl.ntot * K * OCr;
    hipLaunchKernelGGL(reduce_kernel, dim3((unsigned)((nthreads + 255) / 256)), dim3(256), 0, st, rp);
    RMW_CHECK_HIP(hipGetLastError());
  }
}

// RMW_FLAG_CHECK_FINITE: count the non-finite output entries on the stream,
// wait for it and report them as RMW_E_NOTFINITE.
static void check_outputs(const Plan& pl, const double* vel, const double* omg, int k, int64_t stride, char* base,
                          hipStream_t st)
{
  if (!pl.check_finite) return;
  unsigned int* count = (unsigned int*)(base + pl.off_status);
  hipLaunchKernelGGL(zero_count_kernel, dim3(1), dim3(64), 0, st, count);
  RMW_CHECK_HIP(hipGetLastError());
  const int64_t len = 3 * pl.ntot;
  const int64_t grid = std::min<int64_t>(((int64_t)k * len + 255) / 256, 4096);
  for (const double* x : {vel, omg}) {
    if (!x || grid == 0) continue;
    hipLaunchKernelGGL(count_nonfinite_kernel, dim3((unsigned)grid), dim3(256), 0, st, x, (int64_t)k, len, stride,
                       count);
    RMW_CHECK_HIP(hipGetLastError());
  }
  RMW_CHECK_HIP(hipStreamSynchronize(st));
  unsigned int bad = 0;
  RMW_CHECK_HIP(hipMemcpy(&bad, count, sizeof(bad), hipMemcpyDeviceToHost));
  if (bad)
    throw Error(RMW_E_NOTFINITE, std::to_string(bad) + " output entries are inf or NaN (coincident distinct "
                                                       "blobs or non-finite inputs)");
}

// Does an output of the product lie over one of its inputs?
static bool in_place(int mask, int64_t ntot, int k, int64_t stride, const double* r, const double* f, const double* t,
                     const double* vel, const double* omg)
{
  const int64_t len = 3 * ntot, span = (k - 1) * stride + len;
  auto over = [&](const double* out) {
    return overlap(out, span, r, len) || ((mask & (kUF | kWF)) && overlap(out, span, f, span)) ||
           ((mask & (kUT | kWT)) && overlap(out, span, t, span));
  };
  return ((mask & (kUF | kUT)) && over(vel)) || ((mask & (kWF | kWT)) && over(omg));
}

static bool has_images(const double* L)
{
  return L && (L[0] > 0.0 || L[1] > 0.0 || L[2] > 0.0);
}

// Workspace bytes for a call whose lengths L the query does not see: the
// larger of the plans without and with pseudo-periodic images.
static size_t plan_bytes_any_images(int mask, int prec, const int64_t* offsets, int nsys, int k,
                                    const rmw_tuning* tuning, bool ragged, int domain = kDomWall)
{
  const Plan a = make_plan(mask, prec, offsets, nsys, k, tuning, ragged, domain, false);
  const Plan b = make_plan(mask, prec, offsets, nsys, k, tuning, ragged, domain, true);
  return std::max(a.total, b.total);
}

static void run_plan(const Plan& pl, const double* r, const double* f, const double* t, double* vel,
                     double* omg, int k, int64_t ld, double eta, double a, const double* L,
                     const rmw_tuning* tuning, void* ws, size_t ws_bytes, hipStream_t st, bool ragged)
{
  RMW_REQUIRE(ld == 0 || ld >= 3 * pl.ntot, "ld must be 0 or >= 3 n");
  RMW_REQUIRE(ws_bytes >= pl.total, "workspace too small: need " + std::to_string(pl.total) + " bytes");
  if (pl.ntot == 0) return;
  RMW_REQUIRE(r != nullptr && ws != nullptr, "r_vectors / workspace is null");
  RMW_REQUIRE(eta > 0.0 && a > 0.0 && std::isfinite(eta) && std::isfinite(a), "eta and a must be positive");
  const int kmask = kernel_mask(pl.mask);
  RMW_REQUIRE(kmask == pl.mask, "unsupported block combination (use UF, UT, WF, WT, UF|UT, UF|WF, "
                                "UT|WT, WF|WT or all four)");
  const bool NF = (kmask & (kUF | kWF)) != 0, NT = (kmask & (kUT | kWT)) != 0;
  const bool HU = (pl.mask & (kUF | kUT)) != 0, HW = (pl.mask & (kWF | kWT)) != 0;
  RMW_REQUIRE(!((pl.mask & (kUF | kWF)) && f == nullptr), "force is required by the mask");
  RMW_REQUIRE(!((pl.mask & (kUT | kWT)) && t == nullptr), "torque is required by the mask");
  RMW_REQUIRE(!(HU && vel == nullptr), "velocity output is required by the mask");
  RMW_REQUIRE(!(HW && omg == nullptr), "omega output is required by the mask");

  char* base = (char*)ws;
  double Lp[3] = {0, 0, 0};
  int periodic = 0;
  for (int d = 0; d < 3; ++d) {
    double Ld = L ? L[d] : 0.0;
    if (Ld > 0.0) {
      periodic |= 1 << d;
      Lp[d] = Ld / a;
    }
  }
  const double inva = 1.0 / a;
  const double c1 = 1.0 / (8.0 * M_PI * eta * a);
  const double c2 = c1 / a;

  const int64_t stride = ld > 0 ? ld : 3 * pl.ntot;
  // A product in place (an output over an input): every launch that writes
  // outputs reads inputs of blobs that other workgroups write, so the outputs
  // go to the workspace and are copied when all right-hand sides are done.
  const bool staged = in_place(pl.mask, pl.ntot, k, stride, r, f, t, vel, omg);
  const int64_t len = 3 * pl.ntot, out_stride = staged ? len : stride;
  double *out_u = vel, *out_w = omg;
  if (staged) {
    RMW_REQUIRE(pl.stage_bytes > 0, "no room for the outputs of a product in place");
    out_u = (double*)(base + pl.off_stage);
    out_w = out_u + (HU ? k * len : 0);
  }
  if (pl.path == kDirectPath)
    run_direct(pl, r, NF ? f : nullptr, NT ? t : nullptr, HU ? out_u : nullptr, HW ? out_w : nullptr, k, stride,
               out_stride, a, inva, c1, c2, base, st, periodic, Lp);
  else if (pl.path != kOrderedPath)
    run_mutual(pl, r, f, t, out_u, out_w, k, stride, out_stride, a, inva, c1, c2, tuning, base, st, periodic, Lp);
  else
    run_ordered(pl, r, f, t, out_u, out_w, k, stride, out_stride, a, inva, c1, c2, tuning, base, st, periodic, Lp,
                ragged);
  if (staged) {
    if (HU) launch_copy_rows(out_u, len, vel, stride, len, k, st);
    if (HW) launch_copy_rows(out_w, len, omg, stride, len, k, st);
  }
  check_outputs(pl, HU ? vel : nullptr, HW ? omg : nullptr, k, stride, base, st);
}


// ---------------------------------------------------------------------------
// No-allocation entry point: the partial sums live in a fixed device array
// instead of a caller workspace.  Each device holds its own copy of the
// array (for the life of the process); its address on the current device
// is looked up once and kept.  Nothing in it must start at zero: every
// partial-sum slot a reduce reads is written by the pair kernel of the same
// call first.
// ---------------------------------------------------------------------------
static __device__ __align__(256) unsigned char scratch[RMW_NOALLOC_SCRATCH_BYTES];

static void* scratch_address()
{
  static std::mutex mu;
  static void* ptrs[64] = {};
  int dev = 0;
  RMW_CHECK_HIP(hipGetDevice(&dev));
  RMW_REQUIRE(dev >= 0 && dev < 64, "device ordinal out of range");
  std::lock_guard<std::mutex> lk(mu);
  if (ptrs[dev] == nullptr) {
    void* p = nullptr;
    RMW_CHECK_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    RMW_REQUIRE(p != nullptr, "no device address for the scratch array");
    ptrs[dev] = p;
  }
  return ptrs[dev];
}

// The plan of rmw_wall_rpy_apply for these sizes if its partial sums (and, for
// a product in place, its outputs: stage) fit in `cap` bytes; otherwise (unless the tuning requires the symmetric
// kernel) the ordered kernel with source chunks as long as the fit needs,
// and fewer right-hand sides per pass if one chunk of k_group is still too
// large.  Throws RMW_E_LIMIT when nothing fits.
static Plan plan_within(int mask, int prec, int64_t n, int k, const rmw_tuning* tuning, size_t cap, bool periodic,
                        bool stage)
{
  const int64_t off[2] = {0, n};
  const int OC = 3 * (((mask & (kUF | kUT)) ? 1 : 0) + ((mask & (kWF | kWT)) ? 1 : 0));
  const size_t staged = stage ? align_up((size_t)k * n * OC * sizeof(double)) : 0;
  const size_t sums = cap > staged ? cap - staged : 0;
  Plan pl = make_plan(mask, prec, off, 1, k, tuning, false, kDomWall, periodic, stage, sums);
  // (an ordered kernel in the place of a symmetric one takes the chunks below,
  // as short as the array allows: 40000 blobs 2.15 ms, 2.27 with its own)
  if (pl.total <= cap && !pl.over_cap) return pl;
  const bool sym_required = tuning && tuning->symmetric > 0;
  if (!sym_required && sums > 256) {
    rmw_tuning t = tuning ? *tuning : rmw_tuning{};
    t.symmetric = -1;
    for (int g : {4, 2, 1}) {
      if (t.rhs_group != 0 && g > t.rhs_group) continue;
      const int kg = group_k(k, g);
      const double per_chunk = (double)kg * (double)n * OC * sizeof(double);
      const int64_t chunks = (int64_t)std::floor((double)(sums - 256) / per_chunk);
      if (chunks < 1) continue;
      const int64_t len = (n + chunks - 1) / chunks;
      t.chunk_len = std::max<int64_t>(t.chunk_len, (len + kChunkQuantum - 1) / kChunkQuantum * kChunkQuantum);
      t.rhs_group = kg;
      Plan p2 = make_plan(mask, prec, off, 1, k, &t, false, kDomWall, periodic, stage);
      if (p2.total <= cap) return p2;
    }
  }
  throw Error(RMW_E_LIMIT, "rmw_wall_rpy_apply_noalloc: n = " + std::to_string(n) + ", k = " + std::to_string(k) +
                               " needs " + std::to_string(pl.total) + " bytes of partial sums, more than the " +
                               std::to_string((size_t)RMW_NOALLOC_SCRATCH_BYTES) + "-byte scratch array");
}

}  // namespace rmw

// ---------------------------------------------------------------------------
// C ABI
// ---------------------------------------------------------------------------
using namespace rmw;

extern "C" const char* rmw_last_error(void) { return g_last_error.c_str(); }

extern "C" const char* rmw_version(void) { return "rmw_hip 0.1 gfx950"; }

extern "C" int rmw_wall_rpy_workspace_size(int mask, int prec, int64_t n, int k, const rmw_tuning* tuning,
                                           size_t* bytes)
{
  return guarded([&] {
    RMW_REQUIRE(bytes != nullptr, "bytes is null");
    RMW_REQUIRE(n >= 0, "n must be >= 0");
    const int64_t off[2] = {0, n};
    *bytes = plan_bytes_any_images(mask, prec, off, 1, k, tuning, false);
  });
}

extern "C" int rmw_wall_rpy_describe(int mask, int prec, int64_t n, int k, const rmw_tuning* tuning,
                                     int periodic, rmw_plan_info* info)
{
  return guarded([&] {
    RMW_REQUIRE(info != nullptr, "info is null");
    RMW_REQUIRE(n >= 0, "n must be >= 0");
    const int64_t off[2] = {0, n};
    Plan pl = make_plan(mask, prec, off, 1, k, tuning, false, kDomWall, periodic != 0);
    const bool mut = pl.path == kTilesPath || pl.path == kBlocksPath, direct = pl.path == kDirectPath;
    info->symmetric = mut ? 1 : 0;
    info->rhs_group = mut ? pl.kmax_mut : (direct ? pl.kmax_direct : pl.kmax);
    info->chunk_len = mut ? pl.chunk_blocks * 64 : (pl.sys.empty() ? 0 : (direct ? n : pl.sys[0].chunk_len));
    info->work_items = mut ? pl.mut_items : (direct ? pl.direct_wgs : pl.total_items);
    info->workspace_bytes = (int64_t)pl.total;
  });
}

extern "C" int rmw_wall_rpy_apply(int mask, int prec, const double* r_vectors, const double* force,
                                  const double* torque, double* velocity, double* omega, int64_t n, int k,
                                  int64_t ld, double eta, double a, const double* L, const rmw_tuning* tuning,
                                  void* workspace, size_t workspace_bytes, void* stream)
{
  return guarded([&] {
    RMW_REQUIRE(n >= 0, "n must be >= 0");
    const int64_t off[2] = {0, n};
    Plan pl = make_plan(mask, prec, off, 1, k, tuning, false, kDomWall, has_images(L));
    run_plan(pl, r_vectors, force, torque, velocity, omega, k, ld, eta, a, L, tuning, workspace,
             workspace_bytes, (hipStream_t)stream, false);
  });
}

extern "C" int rmw_wall_rpy_apply_noalloc(int mask, int prec, const double* r_vectors, const double* force,
                                          const double* torque, double* velocity, double* omega, int64_t n, int k,
                                          int64_t ld, double eta, double a, const double* L,
                                          const rmw_tuning* tuning, void* stream)
{
  struct NoRecords {
    NoRecords() { tl_no_records = true; }
    ~NoRecords() { tl_no_records = false; }
  } guard;
  return guarded([&] {
    RMW_REQUIRE(n >= 0, "n must be >= 0");
    RMW_REQUIRE(!(tuning && (tuning->flags & RMW_FLAG_CHECK_FINITE)),
                "the finite check waits for the stream; use rmw_wall_rpy_apply for it");
    const bool stage = in_place(mask, n, k, ld > 0 ? ld : 3 * n, r_vectors, force, torque, velocity, omega);
    Plan pl = plan_within(mask, prec, n, k, tuning, RMW_NOALLOC_SCRATCH_BYTES, has_images(L), stage);
    if (pl.ntot == 0) return;
    // the plan may differ from the caller's tuning (longer ordered chunks);
    // run_plan reads only max_wgs and rhs_group from it
    rmw_tuning t = tuning ? *tuning : rmw_tuning{};
    if (pl.path == kOrderedPath) t.rhs_group = pl.kmax;
    run_plan(pl, r_vectors, force, torque, velocity, omega, k, ld, eta, a, L, &t, scratch_address(),
             RMW_NOALLOC_SCRATCH_BYTES, (hipStream_t)stream, false);
  });
}

extern "C" int rmw_mobility_workspace_size(int domain, int mask, int prec, int64_t n, int k,
                                           const rmw_tuning* tuning, size_t* bytes)
{
  return guarded([&] {
    RMW_REQUIRE(bytes != nullptr, "bytes is null");
    RMW_REQUIRE(n >= 0, "n must be >= 0");
    const int64_t off[2] = {0, n};
    *bytes = plan_bytes_any_images(mask, prec, off, 1, k, tuning, false, domain);
  });
}

extern "C" int rmw_mobility_apply(int domain, int mask, int prec, const double* r_vectors, const double* force,
                                  const double* torque, double* velocity, double* omega, int64_t n, int k,
                                  int64_t ld, double eta, double a, const double* L, const rmw_tuning* tuning,
                                  void* workspace, size_t workspace_bytes, void* stream)
{
  return guarded([&] {
    RMW_REQUIRE(n >= 0, "n must be >= 0");
    const int64_t off[2] = {0, n};
    Plan pl = make_plan(mask, prec, off, 1, k, tuning, false, domain, has_images(L));
    run_plan(pl, r_vectors, force, torque, velocity, omega, k, ld, eta, a, L, tuning, workspace,
             workspace_bytes, (hipStream_t)stream, false);
  });
}

// Products between pinned host buffers: a small kernel fetches the inputs (a
// product would read them once per workgroup) and the product writes the
// outputs where the host waits for them (a second kernel that sends them whole
// lines at a time is 1 to 2 us slower up to 8000 blobs and within the noise at
// 14000).  A numpy call of 172 blobs takes 35 us, 70 with torch's copies of
// each array and back; 4000 blobs 77 / 111.
static int64_t host_inputs(int mask, int64_t n)
{
  return 3 * n * (1 + ((mask & (kUF | kWF)) ? 1 : 0) + ((mask & (kUT | kWT)) ? 1 : 0));
}

extern "C" int rmw_mobility_host_workspace_size(int domain, int mask, int prec, int64_t n, const rmw_tuning* tuning,
                                                size_t* bytes)
{
  return guarded([&] {
    RMW_REQUIRE(bytes != nullptr, "bytes is null");
    RMW_REQUIRE(n >= 0, "n must be >= 0");
    const int64_t off[2] = {0, n};
    *bytes = align_up(plan_bytes_any_images(mask, prec, off, 1, 1, tuning, false, domain)) +
             (size_t)host_inputs(mask, n) * sizeof(double);
  });
}

extern "C" int rmw_mobility_apply_host(int domain, int mask, int prec, const double* in, double* out, int64_t n,
                                       double eta, double a, const double* L, const rmw_tuning* tuning,
                                       void* workspace, size_t workspace_bytes, void* stream)
{
  return guarded([&] {
    RMW_REQUIRE(n >= 0, "n must be >= 0");
    const int64_t off[2] = {0, n};
    const Plan pl = make_plan(mask, prec, off, 1, 1, tuning, false, domain, has_images(L));
    const int64_t nin = host_inputs(mask, n);
    const size_t plan_bytes = align_up(pl.total);
    RMW_REQUIRE(workspace_bytes >= plan_bytes + (size_t)nin * sizeof(double), "workspace too small");
    RMW_REQUIRE(in && out && workspace, "in, out and workspace are required");
    if (n == 0) return;
    hipStream_t st = (hipStream_t)stream;
    double* const dev_in = (double*)((char*)workspace + plan_bytes);
    const double *f = nullptr, *t = nullptr, *next = dev_in + 3 * n;
    if (mask & (kUF | kWF)) { f = next; next += 3 * n; }
    if (mask & (kUT | kWT)) t = next;
    double *u = nullptr, *w = nullptr, *onext = out;
    if (mask & (kUF | kUT)) { u = onext; onext += 3 * n; }
    if (mask & (kWF | kWT)) w = onext;
    try {
      launch_copy_rows(in, nin, dev_in, nin, nin, 1, st);
      run_plan(pl, dev_in, f, t, u, w, 1, 0, eta, a, L, tuning, workspace, plan_bytes, st, false);
    } catch (...) {
      (void)hipStreamSynchronize(st);   // the caller's buffers are its own again
      throw;
    }
    RMW_CHECK_HIP(hipStreamSynchronize(st));
  });
}

extern "C" int rmw_wall_rpy_ragged_workspace_size(int mask, int prec, const int64_t* offsets, int nsys, int k,
                                                  const rmw_tuning* tuning, size_t* bytes)
{
  return guarded([&] {
    RMW_REQUIRE(bytes != nullptr && offsets != nullptr && nsys >= 1, "bad arguments");
    *bytes = plan_bytes_any_images(mask, prec, offsets, nsys, k, tuning, true);
  });
}

extern "C" int rmw_wall_rpy_ragged_apply(int mask, int prec, const double* r_vectors, const double* force,
                                         const double* torque, double* velocity, double* omega,
                                         const int64_t* offsets, int nsys, int k, int64_t ld, double eta,
                                         double a, const double* L, const rmw_tuning* tuning, void* workspace,
                                         size_t workspace_bytes, void* stream)
{
  return guarded([&] {
    RMW_REQUIRE(offsets != nullptr && nsys >= 1, "bad offsets");
    Plan pl = make_plan(mask, prec, offsets, nsys, k, tuning, true, kDomWall, has_images(L));
    run_plan(pl, r_vectors, force, torque, velocity, omega, k, ld, eta, a, L, tuning, workspace,
             workspace_bytes, (hipStream_t)stream, true);
  });
}

extern "C" int rmw_profile_enable(int on)
{
  return guarded([&] {
    std::lock_guard<std::mutex> lk(g_prof_mu);
    g_prof_on = on != 0;
  });
}

extern "C" int rmw_profile_collect(int64_t* launches, double* total_ms, double* mean_ms)
{
  return guarded([&] {
    std::vector<ProfRec> recs;
    {
      std::lock_guard<std::mutex> lk(g_prof_mu);
      recs.swap(g_prof);
    }
    double tot = 0.0;
    for (auto& r : recs) {
      RMW_CHECK_HIP(hipEventSynchronize(r.b));
      float ms = 0.f;
      RMW_CHECK_HIP(hipEventElapsedTime(&ms, r.a, r.b));
      tot += ms;
      RMW_CHECK_HIP(hipEventDestroy(r.a));
      RMW_CHECK_HIP(hipEventDestroy(r.b));
    }
    if (launches) *launches = (int64_t)recs.size();
    if (total_ms) *total_ms = tot;
    if (mean_ms) *mean_ms = recs.empty() ? 0.0 : tot / recs.size();
  });
}

extern "C" int rmw_profile_collect_kinds(int64_t* launches, double* total_ms)
{
  return guarded([&] {
    RMW_REQUIRE(launches && total_ms, "launches and total_ms are required");
    std::vector<ProfRec> recs;
    {
      std::lock_guard<std::mutex> lk(g_prof_mu);
      recs.swap(g_prof);
    }
    for (int k = 0; k < kProfKinds; ++k) {
      launches[k] = 0;
      total_ms[k] = 0.0;
    }
    for (auto& r : recs) {
      RMW_CHECK_HIP(hipEventSynchronize(r.b));
      float ms = 0.f;
      RMW_CHECK_HIP(hipEventElapsedTime(&ms, r.a, r.b));
      launches[r.kind] += 1;
      total_ms[r.kind] += ms;
      RMW_CHECK_HIP(hipEventDestroy(r.a));
      RMW_CHECK_HIP(hipEventDestroy(r.b));
    }
  });
}

extern "C" int rmw_profile_pending(int64_t* launches)
{
  return guarded([&] {
    RMW_REQUIRE(launches != nullptr, "launches is null");
    std::lock_guard<std::mutex> lk(g_prof_mu);
    *launches = (int64_t)g_prof.size();
  });
}

extern "C" int rmw_profile_collect_launches(int32_t* kinds, double* ms, int64_t cap, int64_t* launches)
{
  return guarded([&] {
    RMW_REQUIRE(kinds && ms && launches && cap >= 0, "kinds, ms and launches are required");
    std::vector<ProfRec> recs;
    {
      std::lock_guard<std::mutex> lk(g_prof_mu);
      recs.swap(g_prof);
    }
    *launches = (int64_t)recs.size();
    for (size_t i = 0; i < recs.size(); ++i) {
      RMW_CHECK_HIP(hipEventSynchronize(recs[i].b));
      float t = 0.f;
      RMW_CHECK_HIP(hipEventElapsedTime(&t, recs[i].a, recs[i].b));
      if ((int64_t)i < cap) {
        kinds[i] = recs[i].kind;
        ms[i] = t;
      }
      RMW_CHECK_HIP(hipEventDestroy(recs[i].a));
      RMW_CHECK_HIP(hipEventDestroy(recs[i].b));
    }
  });
}

extern "C" int rmw_device_info(int* cu_count, int* clock_khz, int* wavefront, char* arch_name, int arch_len)
{
  return guarded([&] {
    const DeviceProps& p = device_props();
    if (cu_count) *cu_count = p.cu_count;
    if (clock_khz) *clock_khz = p.clock_khz;
    if (wavefront) *wavefront = p.warp;
    if (arch_name && arch_len > 0) {
      std::strncpy(arch_name, p.arch.c_str(), (size_t)arch_len - 1);
      arch_name[arch_len - 1] = '\0';
    }
  });
}
