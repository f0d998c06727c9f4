// Blob-blob soft repulsion: F_i = sum_{j != i} f0(r_ij) (r_j - r_i) over all
// blob pairs (gfx950).
//
// Reference: multi_bodies/forces_numba.py:12-56 (blob_blob_force_numba),
// the different-radii form :75-122 (a = (a_i + a_j) / 2) and the
// neighbour-list form :141-201 (pairs with r <= 2a + 30b only), the same
// force as forces.cpp:11-42 and forces_pycuda.py:24-110, selected by
// set_blob_blob_forces (multi_bodies/multi_bodies_functions.py:249-279).
// The force is minus the gradient of U(r) = eps (1 + (2a - r)/b) for
// r < 2a and eps exp(-(r - 2a)/b) beyond:
//   f0 = -(eps/b) exp(-(r - 2a)/b) / r   (r > 2a),   -(eps/b) / r   (r <= 2a),
// dr = r_j - r_i taken to its minimum image in each periodic direction.
//
// The force has a finite range: beyond 2a + 104 b the FP32 exponential is
// exactly 0, beyond 2a + 746 b the FP64 one, and a cutoff may end it before
// that.  Suspensions of more than a few thousand blobs are therefore sorted
// into cells of that range and every blob visits the 27 cells around it
// ("cells" below); a few thousand blobs take one launch over all pairs
// (force_direct_kernel).  Where the cells would not pay (a range comparable
// with the suspension), the positions do not fit the cell arithmetic (not
// finite, or further out than 2^20 cells) or the radii differ and no cutoff
// bounds the range, all pairs are visited in two launches: a pair kernel and
// a fixed-order reduce.  The force is
// antisymmetric (f0 depends on |dr| and (a_i + a_j) only, and the minimum
// image of -dr is exactly minus that of dr), so the default pair kernel is
// symmetric: each unordered pair of 256-blob tiles is visited once, each
// wave owning 64 target blobs and sweeping 64-source blocks with a rotating
// schedule (at step s lane l takes source (l + s) mod 64) while the
// source-side sum of each source travels with it one lane per step (DPP
// rotation); FP64 partial sums per work item (target side) and per tile
// pair (source side).  The ordered kernel (every target against a chunk of
// sources, one FP64 partial per (chunk, blob)) serves small systems and
// workspaces beyond the symmetric kernel's automatic limit.  Sums carry
// g = e/r; the reduce applies -eps/b.  A blob and its coincident partners
// contribute nothing: r^2 is clamped to 1e-50 (the reference's
// max(r, 1e-25)) and dr = 0.
//
// Precision: the geometry (differences, r, the exponent) and every sum are
// FP64 in both modes.  RMW_PREC_F64 takes 1/r from the FP64 reciprocal
// square root of the pair terms (rsq: <= 1.4e-16 relative) and exp in FP64;
// the other modes take 1/r from the hardware FP64 reciprocal square
// root refined by one Newton step (relative error ~1e-13) and the
// exponential from the hardware FP32 exp2 of the FP64 exponent rounded
// once, which leaves a relative error of ~1e-7 t e^-t per pair with
// t = (r - 2a)/b.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <string>
#include <type_traits>

#include "rmw_accum.h"
#include "rmw_internal.h"
#include "rmw_pair_terms.h"
#include "rmw_tile_pairs.h"

namespace rmw {

constexpr int kFBlock = 256;
// Largest workspace the automatic choice gives the symmetric kernel.
constexpr size_t kFMutAutoBytes = size_t(2) << 30;

struct ForceParams {
  const double* r;
  const double* rad;      // per-blob radius, or null: one radius a
  double a;
  int64_t n;
  double invb;            // 1 / b
  double t2;              // log2(e) / b: exponent scale of the FP32 path
  double cutoff;          // pairs with r > cutoff contribute nothing
  int periodic;           // bit d set when L_d > 0
  double L[3];
  double* partial;        // ordered: [chunk][n][3]; symmetric: target-side slots
  double* part_j;         // symmetric: source-side slots [tri(S, T)][kFBlock][3]
  int64_t n_chunks, chunk_len, total_items;
  int64_t n_t, chunk_tiles;  // symmetric: tiles, source tiles per item
};

// Per-blob radius term kept in LDS / registers: a (FP64 mode) or a t2.
template <bool F64>
__device__ __forceinline__ double radius_term(const ForceParams& p, int64_t j)
{
  const double a = p.rad ? p.rad[j] : p.a;
  return F64 ? a : a * p.t2;
}

// g = f0 / (-eps/b) of a pair at squared distance r2, with A = a_i + a_j
// (FP64 mode) or (a_i + a_j) t2.  FP32 path: 1/r = y0 (1 + (1 - r2 y0^2)/2)
// from the hardware estimate y0, and e = 2^min(t, 0) with 2^0 = 1 exactly
// for the overlap branch.
template <bool F64, bool CUT>
__device__ __forceinline__ double pair_g(const ForceParams& p, double r2, double A)
{
  r2 = fmax(r2, 1e-50);
  double r, inv, e;
  if constexpr (F64) {
    inv = rsq(r2);
    r = r2 * inv;
    e = r > A ? exp(-(r - A) * p.invb) : 1.0;
  } else {
    const double y0 = __builtin_amdgcn_rsq(r2);
    const double h = fma(-r2 * y0, y0, 1.0);
    inv = fma(y0 * h, 0.5, y0);
    r = r2 * inv;
    const float t = (float)fma(-r, p.t2, A);   // -(r - 2a)/b in units of ln 2
    e = (double)__builtin_amdgcn_exp2f(fminf(t, 0.0f));
  }
  const double g = inv * e;
  if constexpr (CUT) return r > p.cutoff ? 0.0 : g;
  return g;
}

// Minimum image of a difference (multi_bodies/forces_numba.py:40-42).
__device__ __forceinline__ void min_image(const ForceParams& p, double& dx, double& dy, double& dz)
{
  if (p.periodic & 1) dx -= image_count(dx, p.L[0]) * p.L[0];
  if (p.periodic & 2) dy -= image_count(dy, p.L[1]) * p.L[1];
  if (p.periodic & 4) dz -= image_count(dz, p.L[2]) * p.L[2];
}

// Ordered pairs: work item = (target tile, source chunk).
template <bool F64, bool CUT>
__device__ __forceinline__ void ordered_items(const ForceParams& p)
{
  __shared__ double s_x[kFBlock], s_y[kFBlock], s_z[kFBlock], s_a[kFBlock];
  const int il = threadIdx.x;

  for (int64_t item = blockIdx.x; item < p.total_items; item += gridDim.x) {
    const int64_t tt = item / p.n_chunks;
    const int64_t ch = item - tt * p.n_chunks;
    const int64_t i = tt * kFBlock + il;
    const bool valid = i < p.n;
    const int64_t gi = valid ? i : 0;
    const double xi = p.r[3 * gi], yi = p.r[3 * gi + 1], zi = p.r[3 * gi + 2];
    const double ai = radius_term<F64>(p, gi);
    double fx = 0.0, fy = 0.0, fz = 0.0;

    const int64_t s_begin = ch * p.chunk_len;
    const int64_t s_end = s_begin + p.chunk_len < p.n ? s_begin + p.chunk_len : p.n;
    for (int64_t s0 = s_begin; s0 < s_end; s0 += kFBlock) {
      const int cnt = (int)(s_end - s0 < kFBlock ? s_end - s0 : kFBlock);
      __syncthreads();
      if (il < cnt) {
        const int64_t j = s0 + il;
        s_x[il] = p.r[3 * j];
        s_y[il] = p.r[3 * j + 1];
        s_z[il] = p.r[3 * j + 2];
        s_a[il] = radius_term<F64>(p, j);
      }
      __syncthreads();
      if (!p.periodic) {
#pragma unroll 4
        for (int j = 0; j < cnt; ++j) {
          const double dx = s_x[j] - xi, dy = s_y[j] - yi, dz = s_z[j] - zi;
          const double g = pair_g<F64, CUT>(p, fma(dx, dx, fma(dy, dy, dz * dz)), ai + s_a[j]);
          fx = fma(g, dx, fx);
          fy = fma(g, dy, fy);
          fz = fma(g, dz, fz);
        }
      } else {
        for (int j = 0; j < cnt; ++j) {
          double dx = s_x[j] - xi, dy = s_y[j] - yi, dz = s_z[j] - zi;
          min_image(p, dx, dy, dz);
          const double g = pair_g<F64, CUT>(p, fma(dx, dx, fma(dy, dy, dz * dz)), ai + s_a[j]);
          fx = fma(g, dx, fx);
          fy = fma(g, dy, fy);
          fz = fma(g, dz, fz);
        }
      }
    }
    if (valid) {
      double* P = p.partial + (ch * p.n + i) * 3;
      P[0] = fx; P[1] = fy; P[2] = fz;
    }
  }
}

template <bool F64, bool CUT>
__global__ __launch_bounds__(kFBlock) void force_kernel(ForceParams p)
{
  ordered_items<F64, CUT>(p);
}

// One step of the symmetric sweep: the pair (target in this lane, source
// at LDS slot js); g is zeroed when !on.
template <bool F64, bool CUT, bool PER, bool MASKED>
__device__ __forceinline__ void mutual_step(const ForceParams& p, const double* s_x, const double* s_y,
                                            const double* s_z, const double* s_a, int js, bool on, double xi,
                                            double yi, double zi, double ai, double& fx, double& fy, double& fz,
                                            double& jx, double& jy, double& jz)
{
  double dx = s_x[js] - xi, dy = s_y[js] - yi, dz = s_z[js] - zi;
  if constexpr (PER) min_image(p, dx, dy, dz);
  double g = pair_g<F64, CUT>(p, fma(dx, dx, fma(dy, dy, dz * dz)), ai + s_a[js]);
  if constexpr (MASKED) g = on ? g : 0.0;
  fx = fma(g, dx, fx);
  fy = fma(g, dy, fy);
  fz = fma(g, dz, fz);
  jx = fma(-g, dx, rol1(jx));
  jy = fma(-g, dy, rol1(jy));
  jz = fma(-g, dz, rol1(jz));
}

// Symmetric pair kernel: work item = (target tile T, run of source tiles
// S >= T); on the diagonal tile only sources above the target are taken.
// Each 64-source block sits twice in LDS ([b][0..63] and [b][64..127]) so
// that lane l reads source (l + s) mod 64 at slot l + s without wrapping.
template <bool F64, bool CUT, bool PER>
__device__ __forceinline__ void mutual_items(const ForceParams& p)
{
  constexpr int NB = kFBlock / 64;
  __shared__ double s_x[NB][128], s_y[NB][128], s_z[NB][128], s_a[NB][128];
  __shared__ double s_jd[NB][3][64];   // per-wave source-side sums of one block
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int il = threadIdx.x;

  for (int64_t item = blockIdx.x; item < p.total_items; item += gridDim.x) {
    const int64_t T = pair_target_tile(item, p.n_t, p.chunk_tiles);
    const int64_t S0 = T + (item - items_before(T, p.n_t, p.chunk_tiles)) * p.chunk_tiles;
    const int64_t S1 = S0 + p.chunk_tiles < p.n_t ? S0 + p.chunk_tiles : p.n_t;
    const int64_t i = T * kFBlock + il;
    const bool valid = i < p.n;
    const bool t_full = (T + 1) * kFBlock <= p.n;
    const int64_t gi = valid ? i : 0;
    const double xi = p.r[3 * gi], yi = p.r[3 * gi + 1], zi = p.r[3 * gi + 2];
    const double ai = radius_term<F64>(p, gi);
    double fx = 0.0, fy = 0.0, fz = 0.0;

    for (int64_t S = S0; S < S1; ++S) {
      const int64_t s0 = S * kFBlock;
      const int cnt = (int)(p.n - s0 < kFBlock ? p.n - s0 : kFBlock);
      __syncthreads();  // the previous tile has been consumed
      {
        double x = 0.0, y = 0.0, z = 0.0, a = 0.0;   // finite stand-ins beyond n: masked below
        if (il < cnt) {
          const int64_t j = s0 + il;
          x = p.r[3 * j]; y = p.r[3 * j + 1]; z = p.r[3 * j + 2];
          a = radius_term<F64>(p, j);
        }
        const int bb = il >> 6, q = il & 63;
        s_x[bb][q] = x; s_y[bb][q] = y; s_z[bb][q] = z; s_a[bb][q] = a;
        s_x[bb][q + 64] = x; s_y[bb][q + 64] = y; s_z[bb][q + 64] = z; s_a[bb][q + 64] = a;
      }
      __syncthreads();
      const bool masked = S == T || !t_full || cnt < kFBlock;
      for (int b = 0; b < NB && 64 * b < cnt; ++b) {
        double jx = 0.0, jy = 0.0, jz = 0.0;
        const double *bx = s_x[b] + lane, *by = s_y[b] + lane, *bz = s_z[b] + lane, *ba = s_a[b] + lane;
        if (!masked) {
#pragma unroll 8
          for (int st = 0; st < 64; ++st)
            mutual_step<F64, CUT, PER, false>(p, bx, by, bz, ba, st, true, xi, yi, zi, ai, fx, fy, fz, jx, jy, jz);
        } else {
          const bool diag = S == T;
#pragma unroll 4
          for (int st = 0; st < 64; ++st) {
            const int jl = 64 * b + ((lane + st) & 63);
            const bool on = valid && jl < cnt && (!diag || jl > il);
            mutual_step<F64, CUT, PER, true>(p, bx, by, bz, ba, st, on, xi, yi, zi, ai, fx, fy, fz, jx, jy, jz);
          }
        }
        // lane l now holds the sum of source (l + 63) mod 64 of the block
        const int jw = (lane + 63) & 63;
        s_jd[wv][0][jw] = jx;
        s_jd[wv][1][jw] = jy;
        s_jd[wv][2][jw] = jz;
        __syncthreads();
        if (il < 64 && 64 * b + il < cnt) {
          double* P = p.part_j + (tri_index(S, T) * kFBlock + 64 * b + il) * 3;
#pragma unroll
          for (int c = 0; c < 3; ++c) P[c] = ((s_jd[0][c][il] + s_jd[1][c][il]) + s_jd[2][c][il]) + s_jd[3][c][il];
        }
        __syncthreads();  // s_jd is free for the next block
      }
    }
    if (valid) {
      double* P = p.partial + (item * kFBlock + il) * 3;
      P[0] = fx; P[1] = fy; P[2] = fz;
    }
  }
}

template <bool F64, bool CUT, bool PER>
__global__ __launch_bounds__(kFBlock) void force_mutual_kernel(ForceParams p)
{
  mutual_items<F64, CUT, PER>(p);
}

// Few blobs, one launch: a workgroup owns kDT targets, its 256 threads share
// the sources (thread t takes t, t + 256, ...), and the 256 partial sums per
// component are added through LDS in a fixed order.  Measured against the
// ordered kernel and its reduce, fp32, open box (us): 9 / 47 at 300 blobs,
// 17 / 56 at 2048.
constexpr int kDT = 4;
template <bool F64, bool CUT>
__device__ __forceinline__ void direct_targets(const ForceParams& p, double scale, double* __restrict__ out)
{
  constexpr int V = 3 * kDT, kRow = kFBlock + 16;
  __shared__ double s_part[V][kRow];
  const int64_t t0 = (int64_t)blockIdx.x * kDT;
  if (t0 >= p.n) return;
  double xi[kDT], yi[kDT], zi[kDT], ai[kDT], f[kDT][3];
#pragma unroll
  for (int q = 0; q < kDT; ++q) {
    const int64_t i = t0 + q < p.n ? t0 + q : p.n - 1;
    xi[q] = p.r[3 * i]; yi[q] = p.r[3 * i + 1]; zi[q] = p.r[3 * i + 2];
    ai[q] = radius_term<F64>(p, i);
    f[q][0] = f[q][1] = f[q][2] = 0.0;
  }
  for (int64_t j = threadIdx.x; j < p.n; j += kFBlock) {
    const double x = p.r[3 * j], y = p.r[3 * j + 1], z = p.r[3 * j + 2];
    const double a = radius_term<F64>(p, j);
#pragma unroll
    for (int q = 0; q < kDT; ++q) {
      double dx = x - xi[q], dy = y - yi[q], dz = z - zi[q];
      min_image(p, dx, dy, dz);
      const double g = pair_g<F64, CUT>(p, fma(dx, dx, fma(dy, dy, dz * dz)), ai[q] + a);
      f[q][0] = fma(g, dx, f[q][0]);
      f[q][1] = fma(g, dy, f[q][1]);
      f[q][2] = fma(g, dz, f[q][2]);
    }
  }
#pragma unroll
  for (int o = 0; o < V; ++o) s_part[o][threadIdx.x] = f[o / 3][o % 3];
  __syncthreads();
  const int o = threadIdx.x >> 4, sub = threadIdx.x & 15;
  if (o < V) {
    double s = 0.0;
#pragma unroll
    for (int m = 0; m < kFBlock / 16; ++m) s += s_part[o][sub + 16 * m];
#pragma unroll
    for (int m = 8; m >= 1; m >>= 1) s += __shfl_xor(s, m, 16);
    if (sub == 0 && t0 + o / 3 < p.n) out[3 * t0 + o] = scale * s;
  }
}

template <bool F64, bool CUT>
__global__ __launch_bounds__(kFBlock) void force_direct_kernel(ForceParams p, double scale, double* __restrict__ out)
{
  direct_targets<F64, CUT>(p, scale, out);
}

// ---------------------------------------------------------------------------
// Cells.  Edges are at least the range of the force (in a periodic direction
// the box divided by a whole number, or one cell when that would give fewer
// than three); a cell's coordinates are hashed into a table of 2 n or more
// buckets, so the table needs no bounds of the suspension, and every stored
// blob carries its cell so that blobs of another cell in the same bucket
// are passed over.  Passes:
//   zero   the bucket counters and the totals;
//   count  cell of every blob, and its place among the bucket's blobs as they
//          arrive;
//   place  first entry of every bucket (one atomic per workgroup: where a
//          bucket lies does not matter);
//   list   the blobs of every bucket, in order of arrival, and an estimate of
//          the pairs the cells will visit, from one blob of every sixteen
//          (the lookups of the 27 cells by one lane for every bucket, in the
//          sort, took 9 us; sixteen lanes to a sampled blob 2: 49 -> 43 us for
//          32768 blobs, 35 -> 28 for 9001 in FP64 in a box);
//   sort   blobs of a bucket by index (the order of arrival differs from run
//          to run, the sums must not), positions gathered;
//   cells  every blob's force, sixteen lanes to a blob.
// If more than a quarter of all ordered pairs would be visited (by the
// estimate, which depends on the blobs and their order alone), or a blob
// does not fit the cell arithmetic, the last launch evaluates all pairs
// instead: as the direct kernel does up to kCellsDirectFallback blobs, by the
// symmetric (or the ordered) kernel, whose reduce follows, beyond.
// ---------------------------------------------------------------------------
struct CellTotals {
  unsigned int cursor;       // entries given out so far
  unsigned int unfit;        // 1: a blob does not fit the cell arithmetic
  unsigned long long pairs;  // pairs the cells will visit
};

struct CellParams {
  double inv_w[3];           // cells per unit length (periodic: per box length)
  int nc[3];                 // periodic direction: number of cells, else 0
  unsigned int mask;         // buckets - 1
  unsigned long long dense;  // pairs beyond which all pairs are visited
  CellTotals* totals;
  unsigned int *count, *start;          // per bucket
  unsigned int *slot, *list, *index;    // per blob
  unsigned long long *cell, *scell;     // per blob: packed cell (unsorted, sorted)
  double4* pos;                         // sorted x, y, z, radius term
};

constexpr int kCellBits = 21, kCellHalf = 1 << (kCellBits - 1);

__device__ __forceinline__ unsigned long long pack_cell(int x, int y, int z)
{
  constexpr unsigned long long m = (1ull << kCellBits) - 1;
  return ((unsigned long long)(unsigned)(x + kCellHalf) & m) | (((unsigned long long)(unsigned)(y + kCellHalf) & m) << kCellBits) |
         (((unsigned long long)(unsigned)(z + kCellHalf) & m) << (2 * kCellBits));
}

__device__ __forceinline__ int cell_coord(unsigned long long c, int d)
{
  return (int)((c >> (d * kCellBits)) & ((1ull << kCellBits) - 1)) - kCellHalf;
}

__device__ __forceinline__ unsigned int bucket_of(unsigned long long c, unsigned int mask)
{
  unsigned long long h = c * 0x9E3779B97F4A7C15ull;
  return (unsigned int)(h >> 32) & mask;
}

// Cell coordinate in direction d; false when it does not fit (the packed
// coordinates and, in a periodic direction, the rounding of x / L that the
// margin of the cell width covers).
__device__ __forceinline__ bool cell_of(const CellParams& c, int d, double x, double L, int& out)
{
  if (c.nc[d] > 0) {
    const double u = x / L;
    if (!(fabs(u) <= 1e5)) return false;
    const int k = (int)((u - floor(u)) * c.nc[d]);
    out = k < c.nc[d] ? k : c.nc[d] - 1;
    return true;
  }
  const double u = floor(x * c.inv_w[d]);
  if (!(fabs(u) < (double)(kCellHalf - 2))) return false;
  out = (int)u;
  return true;
}

// Neighbour q in 0..26 of cell c; false when it repeats another one (a
// direction of a single cell) .
__device__ __forceinline__ bool neighbour(const CellParams& p, unsigned long long c, int q, unsigned long long& out)
{
  int k[3];
  const int off[3] = {q % 3 - 1, (q / 3) % 3 - 1, q / 9 - 1};
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    k[d] = cell_coord(c, d) + off[d];
    if (p.nc[d] == 1) {
      if (off[d] != 0) return false;
      k[d] = 0;
    } else if (p.nc[d] > 0) {
      k[d] = k[d] < 0 ? k[d] + p.nc[d] : (k[d] >= p.nc[d] ? k[d] - p.nc[d] : k[d]);
    }
  }
  out = pack_cell(k[0], k[1], k[2]);
  return true;
}

__global__ __launch_bounds__(256) void cells_zero_kernel(CellParams c)
{
  const unsigned int i = blockIdx.x * 256 + threadIdx.x;
  if (i <= c.mask) c.count[i] = 0u;
  if (i == 0) *c.totals = CellTotals{0u, 0u, 0ull};
}

// Atomics on one counter follow one another at some 12 ns each, which for
// thousands of blobs in a few cells was the time of the whole call: up to eight
// buckets of a wave's blobs take their places by one atomic each (30000 blobs in
// eight cells: 343 us by one atomic per blob, 8 so).
__global__ __launch_bounds__(256) void cells_count_kernel(ForceParams p, CellParams c)
{
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int lane = threadIdx.x & 63;
  bool open = i < p.n;   // a blob without a place
  unsigned int h = 0;
  if (open) {
    int k[3] = {0, 0, 0};
    bool fits = true;
#pragma unroll
    for (int d = 0; d < 3; ++d) fits = cell_of(c, d, p.r[3 * i + d], p.L[d], k[d]) && fits;
    if (!fits) c.totals->unfit = 1u;
    const unsigned long long cell = fits ? pack_cell(k[0], k[1], k[2]) : 0ull;
    c.cell[i] = cell;
    h = bucket_of(cell, c.mask);
  }
  unsigned long long mates = 1ull << lane;   // the lanes that share an atomic, its first lane
  int first = lane;
  for (int t = 0; t < 8; ++t) {
    const unsigned long long left = __ballot(open);
    if (left == 0) break;
    const int f = __ffsll(left) - 1;
    const bool with = open && h == (unsigned int)__shfl((int)h, f, 64);
    const unsigned long long m = __ballot(with);
    if (with) {
      mates = m;
      first = f;
      open = false;
    }
    if (__popcll(m) < 4) break;   // few blobs to a bucket: not worth sharing
  }
  unsigned int base = 0;
  if (i < p.n && lane == first) base = atomicAdd(&c.count[h], (unsigned int)__popcll(mates));
  base = (unsigned int)__shfl((int)base, first, 64);
  if (i < p.n) c.slot[i] = base + (unsigned int)__popcll(mates & ((1ull << lane) - 1));
}

__global__ __launch_bounds__(256) void cells_place_kernel(CellParams c)
{
  __shared__ unsigned int s_wave[4], s_base;
  const unsigned int h = blockIdx.x * 256 + threadIdx.x;
  const unsigned int cnt = h <= c.mask ? c.count[h] : 0u;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  unsigned int sum = cnt;   // inclusive over the wave
  for (int o = 1; o < 64; o <<= 1) {
    const unsigned int v = __shfl_up(sum, o, 64);
    if (lane >= o) sum += v;
  }
  if (lane == 63) s_wave[wv] = sum;
  __syncthreads();
  if (threadIdx.x == 0) s_base = atomicAdd(&c.totals->cursor, s_wave[0] + s_wave[1] + s_wave[2] + s_wave[3]);
  __syncthreads();
  unsigned int before = s_base + sum - cnt;
  for (int w = 0; w < wv; ++w) before += s_wave[w];
  if (h <= c.mask) c.start[h] = before;
}

__global__ __launch_bounds__(256) void cells_list_kernel(ForceParams p, CellParams c)
{
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < p.n) c.list[c.start[bucket_of(c.cell[i], c.mask)] + c.slot[i]] = (unsigned int)i;
  // sixteen lanes look up the 27 cells around one of their sixteen blobs
  unsigned long long visits = 0;
  const int64_t g0 = i & ~(int64_t)15;
  if (g0 < p.n && c.totals->unfit == 0) {
    const int group = p.n - g0 < 16 ? (int)(p.n - g0) : 16;
    const int pick = (int)(((unsigned int)(g0 >> 4) * 2654435761u) >> 28);
    const unsigned long long cell = c.cell[g0 + (pick < group ? pick : 0)];
    for (int q = (int)(i & 15); q < 27; q += 16) {
      unsigned long long nb;
      if (neighbour(c, cell, q, nb)) visits += c.count[bucket_of(nb, c.mask)];
    }
    visits *= group;
  }
  // one atomic per workgroup: they go to one address, one after the other
  __shared__ unsigned long long s_visits[4];
  for (int o = 32; o > 0; o >>= 1) visits += __shfl_down(visits, o, 64);
  if ((threadIdx.x & 63) == 0) s_visits[threadIdx.x >> 6] = visits;
  __syncthreads();
  if (threadIdx.x == 0) atomicAdd(&c.totals->pairs, s_visits[0] + s_visits[1] + s_visits[2] + s_visits[3]);
}

__device__ __forceinline__ bool cells_pay(const CellParams& c)
{
  return c.totals->unfit == 0 && c.totals->pairs <= c.dense;
}

template <bool F64>
__global__ __launch_bounds__(256) void cells_sort_kernel(ForceParams p, CellParams c)
{
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= p.n || !cells_pay(c)) return;
  const unsigned long long cell = c.cell[i];
  const double x = p.r[3 * i], y = p.r[3 * i + 1], z = p.r[3 * i + 2], rad = radius_term<F64>(p, i);
  const unsigned int h = bucket_of(cell, c.mask), s = c.start[h], cnt = c.count[h];
  unsigned int rank = 0;
  for (unsigned int m = 0; m < cnt; m += 8) {   // eight loads in flight
#pragma unroll
    for (unsigned int u = 0; u < 8; ++u) {
      const unsigned int k = m + u < cnt ? m + u : cnt - 1;
      rank += c.list[s + k] < (unsigned int)i && m + u < cnt ? 1u : 0u;
    }
  }
  c.index[s + rank] = (unsigned int)i;
  c.scell[s + rank] = cell;
  c.pos[s + rank] = make_double4(x, y, z, rad);
}

// Force of one blob by the sixteen lanes of its group.  The lanes look up the
// 27 cells together and write the ones with blobs to LDS; then they go over
// all those blobs as one list, sixteen at a time, the next sixteen loaded
// while the present ones are evaluated (cell by cell, eight lanes to a blob and
// nothing in flight meanwhile, the launch took 31.6 us instead of 19.1 at
// 32768 blobs).
constexpr int kCellLanes = 16;
struct CellList {
  unsigned long long id;     // the cell
  unsigned int shift, end;   // entry = place in the list + shift, for places below end
};

template <bool F64, bool CUT, bool PER>
__device__ __forceinline__ void cell_blob(const ForceParams& p, const CellParams& c, double scale,
                                          double* __restrict__ out)
{
  __shared__ CellList s_list[kFBlock / kCellLanes][28];
  const int sub = threadIdx.x & (kCellLanes - 1);
  CellList* list = s_list[threadIdx.x / kCellLanes];
  const int64_t e = ((int64_t)blockIdx.x * kFBlock + threadIdx.x) / kCellLanes;   // sorted entry
  if (e >= p.n) return;   // whole groups leave together
  const double4 own = c.pos[e];
  const unsigned long long cell = c.scell[e];
  unsigned int s[2], cnt[2];
  unsigned long long id[2];
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    const int q = kCellLanes * m + sub;
    s[m] = cnt[m] = 0u;
    id[m] = 0ull;
    if (q < 27 && neighbour(c, cell, q, id[m])) {
      const unsigned int h = bucket_of(id[m], c.mask);
      s[m] = c.start[h];
      cnt[m] = c.count[h];
    }
  }
  // inclusive sums of blobs and of cells with blobs over the group, both
  // rounds of lookups in turn
  unsigned int total = 0, cells = 0;
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    unsigned int b = cnt[m], k = cnt[m] > 0 ? 1u : 0u;
#pragma unroll
    for (int o = 1; o < kCellLanes; o <<= 1) {
      const unsigned int vb = __shfl_up(b, o, kCellLanes), vk = __shfl_up(k, o, kCellLanes);
      if (sub >= o) { b += vb; k += vk; }
    }
    if (cnt[m] > 0) list[cells + k - 1] = CellList{id[m], s[m] - (total + b - cnt[m]), total + b};
    total += __shfl(b, kCellLanes - 1, kCellLanes);
    cells += __shfl(k, kCellLanes - 1, kCellLanes);
  }
  // the group's lanes belong to one wave: its LDS writes are done once they
  // are counted down
  __builtin_amdgcn_wave_barrier();
  __threadfence_block();

  double fx = 0.0, fy = 0.0, fz = 0.0;
  unsigned int f = sub, k = 0;
  CellList at = list[0];   // the blob's own cell has a blob
  double4 o{};
  unsigned long long oc = 0, oid = 0;
  auto fetch = [&] {       // place f of the list
    while (f >= at.end) at = list[++k];
    o = c.pos[f + at.shift];
    oc = c.scell[f + at.shift];
    oid = at.id;
  };
  if (f < total) fetch();
  while (f < total) {
    const double4 now = o;
    const bool in = oc == oid;
    f += kCellLanes;
    if (f < total) fetch();
    double dx = now.x - own.x, dy = now.y - own.y, dz = now.z - own.z;
    if constexpr (PER) min_image(p, dx, dy, dz);
    const double v = pair_g<F64, CUT>(p, fma(dx, dx, fma(dy, dy, dz * dz)), own.w + now.w);
    const double g = in ? v : 0.0;   // a blob of another cell of the bucket
    fx = fma(g, dx, fx);
    fy = fma(g, dy, fy);
    fz = fma(g, dz, fz);
  }
#pragma unroll
  for (int m = kCellLanes / 2; m > 0; m >>= 1) {
    fx += __shfl_xor(fx, m, kCellLanes);
    fy += __shfl_xor(fy, m, kCellLanes);
    fz += __shfl_xor(fz, m, kCellLanes);
  }
  if (sub < 3) out[3 * (int64_t)c.index[e] + sub] = scale * (sub == 0 ? fx : (sub == 1 ? fy : fz));
}

enum : int { kAllDirect, kAllMutual, kAllOrdered };   // how all pairs are evaluated

template <bool F64, bool CUT, bool PER, int ALL>
__global__ __launch_bounds__(kFBlock) void force_cells_kernel(ForceParams p, CellParams c, double scale,
                                                              double* __restrict__ out)
{
  if (cells_pay(c)) cell_blob<F64, CUT, PER>(p, c, scale, out);
  else if constexpr (ALL == kAllDirect) direct_targets<F64, CUT>(p, scale, out);
  else if constexpr (ALL == kAllMutual) mutual_items<F64, CUT, PER>(p);
  else ordered_items<F64, CUT>(p);
}

// Ordered reduce: F = -(eps/b) * (fixed-order sum over chunks).  cells: null,
// or the cells of the call: nothing to do when they have given the forces.
__global__ __launch_bounds__(256) void force_reduce_kernel(const double* __restrict__ partial, int64_t n_chunks,
                                                           int64_t n, double scale, double* __restrict__ out,
                                                           CellParams cells)
{
  if (cells.totals && cells_pay(cells)) return;
  const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (tid >= n * 3) return;
  double s0 = 0.0, s1 = 0.0;
  int64_t ch = 0;
  for (; ch + 2 <= n_chunks; ch += 2) {
    s0 += partial[ch * n * 3 + tid];
    s1 += partial[(ch + 1) * n * 3 + tid];
  }
  if (ch < n_chunks) s0 += partial[ch * n * 3 + tid];
  out[tid] = scale * (s0 + s1);
}

// Symmetric reduce for blob i of tile X: the target-side slots of the items
// of tile X and the source-side slots (X, T) for T = 0..X, split over
// kFRedGroups threads per output, whose sums are added in a fixed order.
constexpr int kFRedGroups = 8, kFRedOut = 256 / kFRedGroups;
__global__ __launch_bounds__(256) void force_mutual_reduce_kernel(const double* __restrict__ part_i,
                                                                  const double* __restrict__ part_j, int64_t n,
                                                                  int64_t n_t, int64_t chunk_tiles, double scale,
                                                                  double* __restrict__ out, CellParams cells)
{
  if (cells.totals && cells_pay(cells)) return;
  __shared__ double part[kFRedGroups][kFRedOut];
  const int g = threadIdx.x / kFRedOut, ol = threadIdx.x - g * kFRedOut;
  const int64_t tid = (int64_t)blockIdx.x * kFRedOut + ol;
  const bool valid = tid < n * 3;
  double s = 0.0;
  if (valid) {
    const int64_t i = tid / 3;
    const int c = (int)(tid - 3 * i);
    const int64_t X = i / kFBlock, l = i - X * kFBlock;
    const int64_t it0 = items_before(X, n_t, chunk_tiles), it1 = items_before(X + 1, n_t, chunk_tiles);
    const int64_t step = (int64_t)kFBlock * 3;
    s = group_strided_sum<kFRedGroups>(part_i + (it0 * kFBlock + l) * 3 + c, it1 - it0, step, g) +
        group_strided_sum<kFRedGroups>(part_j + (tri_index(X, 0) * kFBlock + l) * 3 + c, X + 1, step, g);
  }
  part[g][ol] = s;
  __syncthreads();
  if (g == 0 && valid) {
    double t = part[0][ol];
#pragma unroll
    for (int q = 1; q < kFRedGroups; ++q) t += part[q][ol];
    out[tid] = scale * t;
  }
}

// Up to direct_blobs blobs one launch over all pairs, beyond it the cells
// (unless the tuning names a launch shape: then the kernel it was made for).
// The cells cost 25 to 31 us whatever the size, seven launches; the direct
// kernel's time rises in steps of 1024 blobs (a workgroup per CU).  Rollers
// strip, direct / cells (us): fp32 open 26 / 28 at 5120 blobs, 33 / 28 at 5600,
// periodic 24 / 27 at 3000, 33 / 26 at 3300; FP64 with the cutoff open 22 / 26
// at 3000, 29 / 26 at 3300, periodic 25.5 / 26.5 at 2300, 29 / 26 at 2600.
// Without it the FP64 range (746 Debye lengths) holds most of so small a
// suspension: open 69 / 78 at 6000, 85 / 79 at 6500, periodic 80 / 94 at 5120,
// 104 / 95 at 5600.
static int64_t direct_blobs(bool f64, bool periodic, bool cutoff)
{
  if (!f64) return periodic ? 3072 : 5120;
  if (!cutoff) return periodic ? 5120 : 6144;
  return periodic ? 2304 : 3072;
}
// Blobs up to which all pairs are evaluated by the direct kernel where the cells
// cannot serve the call; direct / symmetric kernel and reduce (us): fp32 open
// 35 / 51 at 6000, 46 / 52 at 7000, 60 / 67 at 8192, periodic 82 / 102 at 6000,
// 110 / 103 at 7000; FP64 open 71 / 87 and 95 / 88, periodic 114 / 136 and
// 152 / 137.
static int64_t direct_fallback(bool f64, bool periodic) { return f64 || periodic ? 6400 : 8192; }
// The same where the cells may turn out not to suit the suspension: the symmetric
// kernel's reduce is then launched whether they do or not, 3 us of 24 when they do.
constexpr int64_t kCellsDirectFallback = 8192;
// Beyond these exponents (r - 2a)/b the exponential is exactly 0.
constexpr double kRangeF64 = 746.0, kRangeF32 = 104.5;

struct ForcePlan {
  bool direct = false, cells = false;
  unsigned int buckets = 0;
  size_t off_cells = 0;
  bool mutual = false;
  int64_t chunk_len = 0, n_chunks = 0, total_items = 0;
  int64_t n_t = 0, chunk_tiles = 0;
  size_t off_pj = 0, bytes = 0;
};

// The cells' arrays at `base` (sizes only when c is null); returns the bytes.
static size_t cells_layout(char* base, int64_t n, unsigned int buckets, CellParams* c)
{
  size_t o = 0;
  auto take = [&](auto*& ptr, size_t count) {
    ptr = reinterpret_cast<std::remove_reference_t<decltype(ptr)>>(base + o);
    o = align_up(o + count * sizeof(*ptr));
  };
  CellParams dummy{};
  CellParams& q = c ? *c : dummy;
  take(q.totals, 1);
  take(q.pos, n);
  take(q.cell, n);
  take(q.scell, n);
  take(q.count, buckets);
  take(q.start, buckets);
  take(q.slot, n);
  take(q.list, n);
  take(q.index, n);
  return o;
}

// Range of the force from the call's own numbers, or 0 when the call does
// not bound it (different radii without a cutoff).
static double force_range(bool f64, bool radii, double a, double b, double cutoff)
{
  const double reach = radii ? 0.0 : 2.0 * a + (f64 ? kRangeF64 : kRangeF32) * b;
  if (cutoff > 0.0 && (reach == 0.0 || cutoff < reach)) return cutoff;
  return reach;
}

static ForcePlan force_plan(int prec, int64_t n, const rmw_tuning* tuning, bool periodic, bool cutoff)
{
  RMW_REQUIRE(prec == RMW_PREC_F32_F64ACC || prec == RMW_PREC_F32_KAHAN || prec == RMW_PREC_F64 ||
                  prec == RMW_PREC_F32_BLOCKED,
              "unknown precision mode");
  RMW_REQUIRE(n >= 0, "n must be >= 0");
  ForcePlan pl;
  const int sym = tuning ? tuning->symmetric : 0;
  const bool shaped = tuning && (tuning->chunk_len > 0 || tuning->max_wgs > 0 || tuning->symmetric != 0);
  // (the workspace query knows neither the box nor the cutoff: it sizes for
  // the cells from the smallest of the limits on)
  pl.direct = !shaped && n > 0 && n <= direct_blobs(prec == RMW_PREC_F64, periodic, cutoff);
  pl.cells = !shaped && !pl.direct && n > 0 && n < (int64_t(1) << 30);
  const int cu = std::max(device_props().cu_count, 1);
  pl.n_t = (n + kFBlock - 1) / kFBlock;
  const int64_t tile_pairs = pl.n_t * (pl.n_t + 1) / 2;
  pl.mutual = n > 0 && sym >= 0 && (sym > 0 || tile_pairs >= cu);
  if (pl.mutual) {
    if (tuning && tuning->chunk_len > 0)
      pl.chunk_tiles = std::max<int64_t>(1, (tuning->chunk_len + kFBlock - 1) / kFBlock);
    else
      pl.chunk_tiles = std::max<int64_t>(1, tile_pairs / (16 * (int64_t)cu));
    pl.total_items = items_before(pl.n_t, pl.n_t, pl.chunk_tiles);
    pl.off_pj = align_up((size_t)pl.total_items * kFBlock * 3 * sizeof(double));
    pl.bytes = pl.off_pj + align_up((size_t)tile_pairs * kFBlock * 3 * sizeof(double));
    if (sym == 0 && pl.bytes > kFMutAutoBytes) pl.mutual = false;
  }
  if (!pl.mutual) {
    int64_t chunk = tuning && tuning->chunk_len > 0 ? tuning->chunk_len : 0;
    if (chunk <= 0) {
      const double c = (double)n * (double)n / (16.0 * cu * kFBlock);
      chunk = std::max<int64_t>(kFBlock, (int64_t)std::ceil(c / 64.0) * 64);
    }
    chunk = std::max<int64_t>(64, (chunk + 63) / 64 * 64);
    if (n > 0) chunk = std::min<int64_t>(chunk, (n + 63) / 64 * 64);
    pl.chunk_len = chunk;
    pl.n_chunks = n > 0 ? (n + chunk - 1) / chunk : 0;
    pl.total_items = pl.n_t * pl.n_chunks;
    pl.off_pj = 0;
    pl.bytes = align_up((size_t)pl.n_chunks * n * 3 * sizeof(double));
  }
  if (pl.direct) {
    pl.total_items = (n + kDT - 1) / kDT;
    pl.bytes = align_up((size_t)n * 3 * sizeof(double));   // the forces of a call in place
  }
  if (pl.cells) {
    pl.buckets = 1024;
    while (pl.buckets < 2 * n) pl.buckets *= 2;
    pl.off_cells = pl.bytes;
    pl.bytes += cells_layout(nullptr, n, pl.buckets, nullptr);
  }
  return pl;
}

template <bool F64, bool CUT>
static void launch_force(bool mutual, const ForceParams& q, int grid, hipStream_t st)
{
  if (!mutual) hipLaunchKernelGGL((force_kernel<F64, CUT>), dim3(grid), dim3(kFBlock), 0, st, q);
  else if (q.periodic) hipLaunchKernelGGL((force_mutual_kernel<F64, CUT, true>), dim3(grid), dim3(kFBlock), 0, st, q);
  else hipLaunchKernelGGL((force_mutual_kernel<F64, CUT, false>), dim3(grid), dim3(kFBlock), 0, st, q);
}

template <bool F64, bool CUT>
static void launch_force_cells(const ForcePlan& pl, const ForceParams& q, const CellParams& c, double scale,
                               double* force, hipStream_t st)
{
  const dim3 b(kFBlock), nb((unsigned)((q.n + 255) / 256)), hb(pl.buckets / 256);
  hipLaunchKernelGGL(cells_zero_kernel, hb, b, 0, st, c);
  hipLaunchKernelGGL(cells_count_kernel, nb, b, 0, st, q, c);
  hipLaunchKernelGGL(cells_place_kernel, hb, b, 0, st, c);
  hipLaunchKernelGGL(cells_list_kernel, nb, b, 0, st, q, c);
  hipLaunchKernelGGL(cells_sort_kernel<F64>, nb, b, 0, st, q, c);
  const bool small = q.n <= kCellsDirectFallback;
  const int64_t all = small ? (q.n + kDT - 1) / kDT : pl.total_items;
  const int64_t wgs = (q.n * kCellLanes + kFBlock - 1) / kFBlock;
  const dim3 g((unsigned)std::min<int64_t>(std::max(wgs, all), (int64_t)INT32_MAX));
  auto run = [&](auto per_c) {
    constexpr bool PER = decltype(per_c)::value;
    if (small) hipLaunchKernelGGL((force_cells_kernel<F64, CUT, PER, kAllDirect>), g, b, 0, st, q, c, scale, force);
    else if (pl.mutual) hipLaunchKernelGGL((force_cells_kernel<F64, CUT, PER, kAllMutual>), g, b, 0, st, q, c, scale, force);
    else hipLaunchKernelGGL((force_cells_kernel<F64, CUT, PER, kAllOrdered>), g, b, 0, st, q, c, scale, force);
  };
  if (q.periodic) run(std::true_type{}); else run(std::false_type{});
}

template <bool F64, bool CUT>
static void launch_any(const ForcePlan& pl, const ForceParams& q, const CellParams& c, bool direct, bool cells,
                       double scale, double* force, int grid, hipStream_t st)
{
  if (direct)
    hipLaunchKernelGGL((force_direct_kernel<F64, CUT>), dim3((unsigned)((q.n + kDT - 1) / kDT)), dim3(kFBlock), 0, st, q,
                       scale, force);
  else if (cells) launch_force_cells<F64, CUT>(pl, q, c, scale, force, st);
  else launch_force<F64, CUT>(pl.mutual, q, grid, st);
}

}  // namespace rmw

using namespace rmw;

extern "C" int rmw_blob_forces_workspace_size(int prec, int64_t n, const rmw_tuning* tuning, size_t* bytes)
{
  return guarded([&] {
    RMW_REQUIRE(bytes != nullptr, "bytes is null");
    *bytes = force_plan(prec, n, tuning, true, true).bytes;
  });
}

extern "C" int rmw_blob_forces_describe(int prec, int64_t n, const rmw_tuning* tuning, rmw_plan_info* info)
{
  return guarded([&] {
    RMW_REQUIRE(info != nullptr, "info is null");
    const ForcePlan pl = force_plan(prec, n, tuning, false, false);
    info->symmetric = pl.mutual && !pl.direct ? 1 : 0;   // with cells: the kernel for dense suspensions
    info->rhs_group = 1;
    info->chunk_len = pl.direct ? n : (pl.mutual ? pl.chunk_tiles * kFBlock : pl.chunk_len);
    info->work_items = pl.total_items;
    info->workspace_bytes = (int64_t)pl.bytes;
  });
}

extern "C" int rmw_blob_forces(int prec, const double* r_vectors, const double* radius_blobs, double* force,
                               int64_t n, double repulsion_strength, double debye_length, double blob_radius,
                               double cutoff, const double* L, const rmw_tuning* tuning, void* workspace,
                               size_t workspace_bytes, void* stream)
{
  return guarded([&] {
    bool boxed = false;
    for (int d = 0; d < 3; ++d) boxed = boxed || (L && L[d] > 0.0);
    const ForcePlan pl = force_plan(prec, n, tuning, boxed, cutoff > 0.0);
    RMW_REQUIRE(workspace_bytes >= pl.bytes, "workspace too small: need " + std::to_string(pl.bytes) + " bytes");
    RMW_REQUIRE(debye_length > 0.0 && std::isfinite(debye_length), "debye_length must be positive");
    RMW_REQUIRE(std::isfinite(repulsion_strength), "repulsion_strength must be finite");
    RMW_REQUIRE(radius_blobs != nullptr || (blob_radius >= 0.0 && std::isfinite(blob_radius)),
                "blob_radius must be >= 0 when no per-blob radii are given");
    RMW_REQUIRE(cutoff >= 0.0, "cutoff must be >= 0 (0: no cutoff)");
    if (n == 0) return;
    RMW_REQUIRE(r_vectors && force && workspace, "r_vectors, force and workspace are required");
    ForceParams q{};
    q.r = r_vectors;
    q.rad = radius_blobs;
    q.a = radius_blobs ? 0.0 : blob_radius;
    q.n = n;
    q.invb = 1.0 / debye_length;
    q.t2 = M_LOG2E / debye_length;
    q.cutoff = cutoff;
    for (int d = 0; d < 3; ++d) {
      const double Ld = L ? L[d] : 0.0;
      q.L[d] = Ld > 0.0 ? Ld : 0.0;
      if (Ld > 0.0) q.periodic |= 1 << d;
    }
    q.partial = (double*)workspace;
    q.part_j = (double*)((char*)workspace + pl.off_pj);
    q.n_chunks = pl.n_chunks;
    q.chunk_len = pl.chunk_len;
    q.total_items = pl.total_items;
    q.n_t = pl.n_t;
    q.chunk_tiles = pl.chunk_tiles;
    int grid = (int)std::min<int64_t>(pl.total_items, (int64_t)INT32_MAX);
    if (tuning && tuning->max_wgs > 0) grid = std::min(grid, tuning->max_wgs);
    hipStream_t st = (hipStream_t)stream;
    ProfRec rec{};
    bool prof = false;
    prof_begin(rec, prof, st, 2);
    const bool cut = cutoff > 0.0, f64 = prec == RMW_PREC_F64;
    const double scale = -repulsion_strength / debye_length;
    // cells at least as wide as the range, with a margin for the rounding of
    // the cell arithmetic
    CellParams c{};
    const double range = force_range(f64, radius_blobs != nullptr, blob_radius, debye_length, cutoff);
    // forces written over an input: the launches below that write them while
    // they read the inputs are not taken, or write to the workspace first
    const bool in_place = overlap(force, 3 * n, r_vectors, 3 * n) || overlap(force, 3 * n, radius_blobs, n);
    bool cells = pl.cells && !in_place && range > 0.0 && std::isfinite(range);
    if (cells) {
      cells_layout((char*)workspace + pl.off_cells, n, pl.buckets, &c);
      c.mask = pl.buckets - 1;
      c.dense = (unsigned long long)n * (unsigned long long)n / 4;
      double share = 1.0;
      for (int d = 0; d < 3; ++d) {
        c.inv_w[d] = 1.0 / (range * (1.0 + 1e-9));
        if (q.L[d] > 0.0) {
          const double k = std::floor(q.L[d] / (range * (1.0 + 1e-9) + 1e-9 * q.L[d]));
          c.nc[d] = k >= 3.0 ? (int)std::min(k, (double)(kCellHalf - 2)) : 1;
          share *= 3.0 / std::max(c.nc[d], 3);
        }
      }
      // a box in which the cells around a blob hold more than a quarter of all
      // blobs: no need to sort to find out
      if (q.L[0] > 0.0 && q.L[1] > 0.0 && share > 0.25) {
        cells = false;
        c = CellParams{};
      }
    }
    // what the cells cannot serve goes the same way as what they turn out not
    // to suit
    const bool direct = pl.direct || (pl.cells && !cells && !in_place && n <= direct_fallback(f64, boxed));
    double* const out = direct && in_place ? (double*)workspace : force;
    if (f64) {
      if (cut) launch_any<true, true>(pl, q, c, direct, cells, scale, out, grid, st);
      else launch_any<true, false>(pl, q, c, direct, cells, scale, out, grid, st);
    } else {
      if (cut) launch_any<false, true>(pl, q, c, direct, cells, scale, out, grid, st);
      else launch_any<false, false>(pl, q, c, direct, cells, scale, out, grid, st);
    }
    RMW_CHECK_HIP(hipGetLastError());
    prof_end(rec, prof, st);
    if (out != force) launch_copy_rows(out, 3 * n, force, 3 * n, 3 * n, 1, st);
    if (direct || (cells && n <= kCellsDirectFallback)) return;
    const dim3 rg((unsigned)((n * 3 + 255) / 256)), rb(256);
    if (pl.mutual)
      hipLaunchKernelGGL(force_mutual_reduce_kernel, dim3((unsigned)((n * 3 + kFRedOut - 1) / kFRedOut)), rb, 0, st,
                         q.partial, q.part_j, n, pl.n_t, pl.chunk_tiles, scale, force, c);
    else
      hipLaunchKernelGGL(force_reduce_kernel, rg, rb, 0, st, q.partial, pl.n_chunks, n, scale, force, c);
    RMW_CHECK_HIP(hipGetLastError());
  });
}
