// Leaf-block solve of the preconditioner (Mobility/ReducedSolve.m:164-209):
// for every target leaf, solve K(leaf sources -> leaf targets) x = v, or in
// NEAREST mode (K(fine -> targets) kron(NN_leaf, I3)) x = v (ReducedSolve.m
// :170-187).  The 3n x 3n blocks are formed and LU-factored with partial
// pivoting once per tree on the GPU (panel by panel, all leaves in a launch),
// and each block's inverse is formed from its factors; each solve is then one
// block-diagonal matrix-vector product.  MATLAB's mldivide would use
// Cholesky on the symmetric non-NEAREST blocks; both give the solution up
// to rounding (relative error of order cond(A) times the FP64 epsilon).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>
#include <vector>

#include "nnk_fmm.hpp"
#include "nnk_kernels.hpp"

namespace nnk {

struct RedArgs {
  const int32_t *leaves;
  const int32_t *tgt_ptr;
  const double *tgt_pos;
  const int32_t *tgt_out;
  const int32_t *src_ptr;
  const double *src_pos;
  const int64_t *ctr_ptr;   // NEAREST: contributions per source instance
  const int32_t *ctr_col;
  const double *ctr_w;
  const int32_t *ord2loc;   // target ordinal -> index within its leaf
  const int64_t *off;       // block offset (doubles) per leaf slot
  double *blk;
  int32_t *piv;             // 3n pivots per leaf at off3[leaf]
  int32_t *perm;            // the pivots as one permutation (same offsets)
  const int64_t *poff;
  double e2, c;
  int nearest;
};

// form the leaf block: rows 3t+a (targets), columns 3j+b (the leaf's coarse
// points in target order); block stored row-major
__global__ __launch_bounds__(256) void k_red_form(RedArgs a) {
  const int li = blockIdx.x;
  const int n = a.leaves[li];
  const int tb = a.tgt_ptr[n], nt = a.tgt_ptr[n + 1] - tb;
  const int n3 = 3 * nt;
  double *A = a.blk + a.off[li];
  for (int i = threadIdx.x; i < n3 * n3; i += 256) A[i] = 0.0;
  __syncthreads();
  const int sb = a.src_ptr[n], se = a.src_ptr[n + 1];
  for (int t = threadIdx.x; t < nt; t += 256) {
    const double *tp = a.tgt_pos + 3 * (size_t)(tb + t);
    double *row = A + (size_t)(3 * t) * n3;
    for (int s = sb; s < se; s++) {
      const double *sp = a.src_pos + 3 * (size_t)s;
      double rx = tp[0] - sp[0], ry = tp[1] - sp[1], rz = tp[2] - sp[2];
      double r2 = rx * rx + ry * ry + rz * rz;
      double inv = rsqrt(r2 + a.e2);
      double w3 = a.c * inv * inv * inv;
      double iso = r2 + 2.0 * a.e2;
      double r[3] = {rx, ry, rz};
      if (!a.nearest) {
        const int j = s - sb;  // sources and targets share the leaf order
        for (int p = 0; p < 3; p++)
          for (int q = 0; q < 3; q++)
            row[(size_t)p * n3 + 3 * j + q] = (r[p] * r[q] + (p == q ? iso : 0.0)) * w3;
      } else {
        for (int64_t e = a.ctr_ptr[s]; e < a.ctr_ptr[s + 1]; e++) {
          const int j = a.ord2loc[a.ctr_col[e]];
          const double w = a.ctr_w[e] * w3;
          for (int p = 0; p < 3; p++)
            for (int q = 0; q < 3; q++)
              row[(size_t)p * n3 + 3 * j + q] += (r[p] * r[q] + (p == q ? iso : 0.0)) * w;
        }
      }
    }
  }
}

// In-place LU with partial pivoting (first maximal |a_ik|), blocked
// right-looking (the order of LAPACK's getrf), three launches per 32-column
// panel for every leaf at once: k_red_lu_panel (one workgroup per leaf)
// factors the panel; k_red_lu_rows (a thread per column) applies its row
// interchanges to the other columns and solves the panel's rows of U right of
// it with its unit lower triangle; k_red_lu_update subtracts the rank-32
// product from every 64 x 64 tile of the trailing matrix.
// While more than kLuRows rows are left, k_red_lu_panel_mem does the work of
// the first two in memory.
// Measured for ten squirmers in a box (blocks up to 832 rows, 26 panels), all
// panels: panel and rows 6.5 -> 2.0 ms (43 to 80 and 15 us each), updates
// 1.0 -> 0.43 ms.
constexpr int kLuThreads = 512, kLuNB = 32, kLuT = 64, kLuRows = 1024;
__global__ __launch_bounds__(kLuThreads) void k_red_lu_panel_mem(RedArgs a, int k0) {
  const int li = blockIdx.x;
  const int n = a.leaves[li];
  const int n3 = 3 * (a.tgt_ptr[n + 1] - a.tgt_ptr[n]);
  if (k0 >= n3) return;  // the whole workgroup
  double *A = a.blk + a.off[li];
  int32_t *piv = a.piv + a.poff[li];
  __shared__ double sv[kLuThreads];
  __shared__ int si[kLuThreads];
  const int tid = threadIdx.x;
  const int k1 = min(k0 + kLuNB, n3);
  for (int k = k0; k < k1; k++) {
    double best = -1.0;
    int bi = n3;
    for (int i = k + tid; i < n3; i += kLuThreads) {
      const double v = fabs(A[(size_t)i * n3 + k]);
      if (v > best) { best = v; bi = i; }
    }
    sv[tid] = best;
    si[tid] = bi;
    __syncthreads();
    for (int st = kLuThreads / 2; st > 0; st >>= 1) {
      if (tid < st) {
        const double v2 = sv[tid + st];
        const int i2 = si[tid + st];
        if (v2 > sv[tid] || (v2 == sv[tid] && i2 < si[tid])) {
          sv[tid] = v2;
          si[tid] = i2;
        }
      }
      __syncthreads();
    }
    const int p = si[0] < n3 ? si[0] : k;   // a column of NaN has no maximum
    if (tid == 0) piv[k] = p;
    if (p != k)
      for (int jj = tid; jj < n3; jj += kLuThreads) {
        const double t = A[(size_t)k * n3 + jj];
        A[(size_t)k * n3 + jj] = A[(size_t)p * n3 + jj];
        A[(size_t)p * n3 + jj] = t;
      }
    __syncthreads();
    const double d = A[(size_t)k * n3 + k];
    if (d != 0.0)
      for (int i = k + 1 + tid; i < n3; i += kLuThreads) A[(size_t)i * n3 + k] /= d;
    __syncthreads();
    const int w = k1 - k - 1;  // panel columns right of k
    if (w > 0) {
      const int m = n3 - k - 1;
      for (int idx = tid; idx < m * w; idx += kLuThreads) {
        const int i = k + 1 + idx / w, jj = k + 1 + idx % w;
        A[(size_t)i * n3 + jj] -= A[(size_t)i * n3 + k] * A[(size_t)k * n3 + jj];
      }
    }
    __syncthreads();
  }
  if (k1 >= n3) return;
  const int m = n3 - k1;  // trailing size
  // U12 = L11^-1 A12 (rows k0..k1-1, columns k1..)
  for (int k = k0; k < k1 - 1; k++) {
    const int h = k1 - k - 1;
    for (int idx = tid; idx < h * m; idx += kLuThreads) {
      const int i = k + 1 + idx / m, jj = k1 + idx % m;
      A[(size_t)i * n3 + jj] -= A[(size_t)i * n3 + k] * A[(size_t)k * n3 + jj];
    }
    __syncthreads();
  }
}

// the largest value of a wavefront, in every lane
__device__ __forceinline__ double wave_max(double v) {
  auto step = [&](auto ctrl) {
    constexpr int c = decltype(ctrl)::value;   // row_shr 1, 2, 4, 8, row_bcast 15, 31: lane 63 ends with all
    const int lo = __double2loint(v), hi = __double2hiint(v);
    const int l2 = __builtin_amdgcn_update_dpp(lo, lo, c, 0xf, 0xf, false);
    const int h2 = __builtin_amdgcn_update_dpp(hi, hi, c, 0xf, 0xf, false);
    v = fmax(v, __hiloint2double(h2, l2));
  };
  step(std::integral_constant<int, 0x111>{});
  step(std::integral_constant<int, 0x112>{});
  step(std::integral_constant<int, 0x114>{});
  step(std::integral_constant<int, 0x118>{});
  step(std::integral_constant<int, 0x142>{});
  step(std::integral_constant<int, 0x143>{});
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), 63),
                          __builtin_amdgcn_readlane(__double2loint(v), 63));
}

// The panel in registers, a thread per row (at most T rows are left): per
// column one reduction for the pivot and one exchange of two rows through LDS,
// the eliminations from registers.
template <int T>
__global__ __launch_bounds__(T) void k_red_lu_panel(RedArgs a, int k0) {
  constexpr int NW = T / 64, NB = kLuNB;
  const int li = blockIdx.x;
  const int n = a.leaves[li];
  const int n3 = 3 * (a.tgt_ptr[n + 1] - a.tgt_ptr[n]);
  if (k0 >= n3) return;  // the whole workgroup
  int32_t *piv = a.piv + a.poff[li];
  __shared__ double bv[2][NW], rowp[NB], rowk[NB];
  __shared__ int bi[2][NW];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int m = n3 - k0, w = min(NB, m);
  const bool own = tid < m;
  double *row = a.blk + a.off[li] + (size_t)(k0 + min(tid, m - 1)) * n3 + k0;
  double x[NB];
#pragma unroll
  for (int c = 0; c < NB; c++) x[c] = c < w ? row[c] : 0.0;
#pragma unroll
  for (int k = 0; k < NB; k++) {
    if (k < w) {   // uniform
      double v = own && tid >= k ? fabs(x[k]) : -1.0;
      if (!(v >= 0.0)) v = -1.0;   // NaN is no pivot
      const double wm = wave_max(v);
      const int first = __ffsll(__ballot(v == wm)) - 1;
      if (lane == 0) {
        bv[k & 1][wave] = wm;
        bi[k & 1][wave] = wave * 64 + first;
      }
      __syncthreads();
      const double g = bv[k & 1][min(lane, NW - 1)];   // the same row order in every wavefront: the first maximum
      const double gm = wave_max(g);
      const int p = gm < 0.0 ? k : bi[k & 1][__ffsll(__ballot(g == gm)) - 1];
      if (tid == p)
#pragma unroll
        for (int c = 0; c < NB; c++) rowp[c] = x[c];
      if (tid == k)
#pragma unroll
        for (int c = 0; c < NB; c++) rowk[c] = x[c];
      if (tid == 0) piv[k0 + k] = k0 + p;
      __syncthreads();
      if (tid == p || tid == k) {
#pragma unroll
        for (int c = 0; c < NB; c++) x[c] = tid == k ? rowp[c] : rowk[c];
      }
      if (tid > k) {
        const double d = rowp[k];
        if (d != 0.0) x[k] /= d;
#pragma unroll
        for (int c = k + 1; c < NB; c++) x[c] -= x[k] * rowp[c];
      }
    }
  }
  if (own)
#pragma unroll
    for (int c = 0; c < NB; c++)
      if (c < w) row[c] = x[c];
}

// The panel's row interchanges in the columns outside it, as one permutation
// of its rows and the (at most 32) rows they were exchanged with, and U12 =
// L11^-1 A12 right of it: a thread per column, its rows in registers.
__global__ __launch_bounds__(256) void k_red_lu_rows(RedArgs a, int k0) {
  constexpr int NB = kLuNB;
  const int li = blockIdx.x;
  const int n = a.leaves[li];
  const int n3 = 3 * (a.tgt_ptr[n + 1] - a.tgt_ptr[n]);
  if (k0 >= n3 || (int)blockIdx.y * 256 >= n3) return;  // the whole workgroup
  const int w = min(NB, n3 - k0), tid = threadIdx.x;
  double *A = a.blk + a.off[li] + (size_t)k0 * n3;      // row 0: the panel's first
  __shared__ double L[NB][NB + 1];
  __shared__ int pv[NB], slot[NB], cur[2 * NB];
  if (tid < NB) pv[tid] = tid < w ? a.piv[a.poff[li] + k0 + tid] - k0 : tid;
  for (int idx = tid; idx < NB * NB; idx += 256) {
    const int r = idx / NB, c = idx % NB;
    L[r][c] = r < w && c < w ? A[(size_t)r * n3 + k0 + c] : 0.0;
  }
  __syncthreads();
  // slots: the panel's rows, then, for exchange i with a row below, NB + (the
  // first exchange with that row); cur[slot] is the row whose entries the
  // slot's row ends with
  if (tid < NB) {
    const int p = pv[tid];
    int sl = p;
    if (p >= NB) {
      int f = 0;
      while (pv[f] != p) f++;
      sl = NB + f;
    }
    slot[tid] = sl;
    cur[tid] = tid;
    cur[NB + tid] = p;
  }
  __syncthreads();
  if (tid == 0)
    for (int i = 0; i < w; i++) {
      const int t = cur[i], s = slot[i];
      cur[i] = cur[s];
      cur[s] = t;
    }
  __syncthreads();
  const int j = blockIdx.y * 256 + tid;
  if (j >= n3 || (j >= k0 && j < k0 + w)) return;
  double x[NB], y[NB];
#pragma unroll
  for (int i = 0; i < NB; i++) {
    x[i] = i < w ? A[(size_t)cur[i] * n3 + j] : 0.0;
    y[i] = slot[i] == NB + i ? A[(size_t)cur[NB + i] * n3 + j] : 0.0;
  }
#pragma unroll
  for (int i = 0; i < NB; i++)
    if (slot[i] == NB + i) A[(size_t)pv[i] * n3 + j] = y[i];
  if (j >= k0 + w) {
#pragma unroll
    for (int k = 0; k < NB; k++)
#pragma unroll
      for (int i = k + 1; i < NB; i++) x[i] -= L[i][k] * x[k];
  }
#pragma unroll
  for (int i = 0; i < NB; i++)
    if (i < w) A[(size_t)i * n3 + j] = x[i];
}

typedef double rd4 __attribute__((ext_vector_type(4)));

// A22 -= L21 U12 after the panel at k0: workgroup (leaf, t) updates tile t
// of the leaf's trailing matrix (row-major over its ceil(m / 64)^2 tiles), a
// wavefront 32 x 32 of it on the FP64 matrix cores, operands from memory.
__global__ __launch_bounds__(256, 2) void k_red_lu_update(RedArgs a, int k0) {
  const int li = blockIdx.x;
  const int n = a.leaves[li];
  const int n3 = 3 * (a.tgt_ptr[n + 1] - a.tgt_ptr[n]);
  const int k1 = k0 + kLuNB;
  if (k1 >= n3) return;  // the whole workgroup
  const int m = n3 - k1, nt = (m + kLuT - 1) / kLuT;
  const int t = blockIdx.y;
  if (t >= nt * nt) return;
  double *A = a.blk + a.off[li];
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int lr = lane & 15, lk = lane >> 4;
  const int r0 = k1 + (t / nt) * kLuT + (wave >> 1) * 32, c0 = k1 + (t % nt) * kLuT + (wave & 1) * 32;
  if (r0 >= n3 || c0 >= n3) return;   // (no barrier below)
  rd4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int c = 0; c < 2; c++) acc[i][c] = rd4{0, 0, 0, 0};
  // rows and columns past n3 repeat the last one and are not stored
  const double *Lp[2] = {A + (size_t)min(r0 + lr, n3 - 1) * n3 + k0, A + (size_t)min(r0 + 16 + lr, n3 - 1) * n3 + k0};
  const double *Up[2] = {A + (size_t)k0 * n3 + min(c0 + lr, n3 - 1), A + (size_t)k0 * n3 + min(c0 + 16 + lr, n3 - 1)};
#pragma unroll
  for (int h = 0; h < kLuNB; h += 16) {
    double f[2][4], u[2][4];
#pragma unroll
    for (int s = 0; s < 4; s++)
#pragma unroll
      for (int i = 0; i < 2; i++) {
        f[i][s] = Lp[i][h + 4 * lk + s];
        u[i][s] = Up[i][(size_t)(h + 4 * lk + s) * n3];
      }
#pragma unroll
    for (int s = 0; s < 4; s++)
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int c = 0; c < 2; c++)
          acc[i][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(f[i][s], u[c][s], acc[i][c], 0, 0, 0);
  }
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int c = 0; c < 2; c++)
#pragma unroll
      for (int s = 0; s < 4; s++) {
        const int r = r0 + 16 * i + lk + 4 * s, q = c0 + 16 * c + lr;
        if (r < n3 && q < n3) A[(size_t)r * n3 + q] -= acc[i][c][s];
      }
}

// the row interchanges of each leaf's LU, applied in order to the identity:
// perm[i] is the row of the right-hand side that lands in position i
__global__ void k_red_perm(RedArgs a, int nleaves) {
  const int li = blockIdx.x * blockDim.x + threadIdx.x;
  if (li >= nleaves) return;
  const int n = a.leaves[li];
  const int n3 = 3 * (a.tgt_ptr[n + 1] - a.tgt_ptr[n]);
  const int32_t *piv = a.piv + a.poff[li];
  int32_t *perm = a.perm + a.poff[li];
  for (int i = 0; i < n3; i++) perm[i] = i;
  for (int k = 0; k < n3; k++) {
    const int p = piv[k];
    const int32_t t = perm[k];
    perm[k] = perm[p];
    perm[p] = t;
  }
}

// The inverses of the 32 x 32 diagonal tiles of each leaf's factors (unit
// lower and upper triangle, row-major, padded with the identity), D[2 I] and
// D[2 I + 1] of block row I: one wavefront per tile pair, a lane per column.
constexpr int kInvB = 32;
__global__ __launch_bounds__(64) void k_red_diag(RedArgs a, const int64_t *__restrict__ doff, double *__restrict__ D) {
  constexpr int B = kInvB;
  __shared__ double T[B][B + 1];
  const int li = blockIdx.x;
  const int n = a.leaves[li];
  const int n3 = 3 * (a.tgt_ptr[n + 1] - a.tgt_ptr[n]);
  const int i0 = blockIdx.y * B;
  if (i0 >= n3) return;
  const double *A = a.blk + a.off[li];
  const int lane = threadIdx.x, c = lane & 31;
  for (int r = lane >> 5; r < B; r += 2)
    T[r][c] = i0 + r < n3 && i0 + c < n3 ? A[(size_t)(i0 + r) * n3 + i0 + c] : (r == c ? 1.0 : 0.0);
  __syncthreads();
  double x[B];
  double *O = D + doff[li] + (size_t)(2 * blockIdx.y + (lane >> 5)) * B * B + c;
  if (lane < 32) {
#pragma unroll
    for (int r = 0; r < B; r++) {
      double t = r == c ? 1.0 : 0.0;
#pragma unroll
      for (int q = 0; q < r; q++) t -= T[r][q] * x[q];
      x[r] = t;
    }
  } else {
#pragma unroll
    for (int r = B - 1; r >= 0; r--) {
      double t = r == c ? 1.0 : 0.0;
#pragma unroll
      for (int q = r + 1; q < B; q++) t -= T[r][q] * x[q];
      x[r] = t / T[r][r];
    }
  }
#pragma unroll
  for (int r = 0; r < B; r++) O[(size_t)r * B] = x[r];
}

// The inverse of each leaf block from its LU factors (set-up only), column-
// major in W (W[j n3 + i] = (A^-1)_ij = U^-1 L^-1 P).  A wavefront owns 16
// columns and walks the rows in blocks of 32, forward with the unit lower
// triangle, then back with the upper one: the solved blocks times the factor
// tiles on the FP64 matrix cores (operands straight from memory, one tile
// ahead), then the diagonal tile's inverse times the block, whose accumulator
// registers are the B operand as they are (register r holds row lk + 4 r).
// No barrier: the wavefronts are independent, four neighbours share a
// workgroup for the factors' sake.  What bounds it is the chain of (n3 / 32)^2
// tiles of 16 MFMAs per wavefront.
// Measured for ten squirmers in a box (blocks up to 832 rows): 5.5 ms with
// scalar sums and two transposes of 0.86 ms, now 2.2 ms.
__global__ __launch_bounds__(256, 2) void k_red_inv(RedArgs a, const int64_t *__restrict__ doff,
                                                    const double *__restrict__ D, double *W) {
  constexpr int B = kInvB;
  const int li = blockIdx.x;
  const int n = a.leaves[li];
  const int n3 = 3 * (a.tgt_ptr[n + 1] - a.tgt_ptr[n]);
  const int lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
  const int j0 = (blockIdx.y * 4 + __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6)) * 16;
  if (j0 >= n3) return;   // (no barrier below)
  const int j = j0 + lr, jc = min(j, n3 - 1);
  const double *A = a.blk + a.off[li];   // row-major factors
  const double *Dl = D + doff[li];
  const int32_t *perm = a.perm + a.poff[li];
  double *X = W + a.off[li] + (size_t)jc * n3;   // a lane past the last column computes a copy and stores nothing
  const int nb = (n3 + B - 1) / B;
  struct Tile { double f[2][2][4], x[2][4]; };
  // factor tile (rows i0 .., columns of block K) and the solved block K;
  // entries past n3 only in the last block
  auto fetch = [&](int i0, int K, Tile &t) {
    const int k0 = K * B;
    if (k0 + B <= n3) {
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const int k = k0 + 16 * h + 4 * lk;
#pragma unroll
        for (int r = 0; r < 2; r++)
#pragma unroll
          for (int s = 0; s < 4; s++) t.f[r][h][s] = A[(size_t)min(i0 + 16 * r + lr, n3 - 1) * n3 + k + s];
#pragma unroll
        for (int s = 0; s < 4; s++) t.x[h][s] = X[k + s];
      }
    } else {
#pragma unroll
      for (int h = 0; h < 2; h++)
#pragma unroll
        for (int s = 0; s < 4; s++) {
          const int k = k0 + 16 * h + 4 * lk + s, kc = min(k, n3 - 1);
#pragma unroll
          for (int r = 0; r < 2; r++) t.f[r][h][s] = A[(size_t)min(i0 + 16 * r + lr, n3 - 1) * n3 + kc];
          const double v = X[kc];
          t.x[h][s] = k < n3 ? v : 0.0;
        }
    }
  };
  rd4 acc[2];
  auto sub = [&](const Tile &t) {
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
      for (int s = 0; s < 4; s++)
#pragma unroll
        for (int r = 0; r < 2; r++)
          acc[r] = __builtin_amdgcn_mfma_f64_16x16x4f64(t.f[r][h][s], -t.x[h][s], acc[r], 0, 0, 0);
  };
  // acc -= sum over blocks K in [ka, kb) of tile (i0, K) times block K
  auto sweep = [&](int i0, int ka, int kb) {
    if (ka >= kb) return;
    Tile t0, t1;
    fetch(i0, ka, t0);
#pragma unroll 1
    for (int K = ka; K < kb; K += 2) {
      fetch(i0, min(K + 1, kb - 1), t1);
      sub(t0);
      if (K + 1 == kb) break;
      fetch(i0, min(K + 2, kb - 1), t0);
      sub(t1);
    }
  };
  // block row I = D^-1 acc, stored to X
  auto solve = [&](int I, int upper) {
    const int i0 = I * B;
    const double *T = Dl + (size_t)(2 * I + upper) * B * B;
    rd4 o[2] = {rd4{0, 0, 0, 0}, rd4{0, 0, 0, 0}};
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
      for (int s = 0; s < 4; s++) {
        const int k = 16 * h + 4 * s + lk;
        const double v = i0 + k < n3 ? acc[h][s] : 0.0;
#pragma unroll
        for (int r = 0; r < 2; r++)
          o[r] = __builtin_amdgcn_mfma_f64_16x16x4f64(T[(16 * r + lr) * B + k], v, o[r], 0, 0, 0);
      }
    if (j < n3)
#pragma unroll
      for (int r = 0; r < 2; r++)
#pragma unroll
        for (int s = 0; s < 4; s++)
          if (i0 + 16 * r + lk + 4 * s < n3) X[i0 + 16 * r + lk + 4 * s] = o[r][s];
    // the next blocks read these rows through other lanes of this wavefront
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
  };
  for (int I = 0; I < nb; I++) {  // L y = P e_j
#pragma unroll
    for (int r = 0; r < 2; r++)
#pragma unroll
      for (int s = 0; s < 4; s++) {
        const int i = I * B + 16 * r + lk + 4 * s;
        acc[r][s] = i < n3 && perm[min(i, n3 - 1)] == j ? 1.0 : 0.0;
      }
    sweep(I * B, 0, I);
    solve(I, 0);
  }
  for (int I = nb - 1; I >= 0; I--) {  // U x = y
#pragma unroll
    for (int r = 0; r < 2; r++)
#pragma unroll
      for (int s = 0; s < 4; s++) acc[r][s] = X[min(I * B + 16 * r + lk + 4 * s, n3 - 1)];
    sweep(I * B, I + 1, nb);
    solve(I, 1);
  }
}

// x = A^-1 v for each leaf with the column-major inverse
// (Inv[j n3 + i] = (A^-1)_ij), one pass over the inverses, in three shapes
// (reduced_solve has the lines between them).
// Few large blocks: a workgroup takes 64 rows of a leaf (lane = row, so a
// column's rows are read coalesced), its wavefronts an eighth of the columns
// each, the sums added in wavefront order.  A thread walking a whole row alone
// has one load in flight per 500 ns.
// Measured for ten squirmers in a box (blocks up to 832 rows): 71 -> 20 us.
constexpr int kRedApplyWaves = 8;
__global__ __launch_bounds__(64 * kRedApplyWaves) void k_red_apply(RedArgs a, const double *__restrict__ v,
                                                                   double *__restrict__ x) {
  extern __shared__ double b[];
  __shared__ double part[kRedApplyWaves][64];
  const int li = blockIdx.x;
  const int n = a.leaves[li];
  const int tb = a.tgt_ptr[n], nt = a.tgt_ptr[n + 1] - tb;
  const int n3 = 3 * nt;
  const int i0 = blockIdx.y * 64;
  if (i0 >= n3) return;  // the whole workgroup
  const double *Inv = a.blk + a.off[li];
  for (int i = threadIdx.x; i < n3; i += 64 * kRedApplyWaves)
    b[i] = v[3 * (size_t)a.tgt_out[tb + i / 3] + i % 3];
  __syncthreads();
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, i = i0 + lane;
  const int j1 = n3 * (w + 1) / kRedApplyWaves;
  const double *col = Inv + min(i, n3 - 1);
  double acc[4] = {0, 0, 0, 0};
  int j = n3 * w / kRedApplyWaves;
  for (; j + 8 <= j1; j += 8) {
    double t[8];
#pragma unroll
    for (int k = 0; k < 8; k++) t[k] = col[(size_t)(j + k) * n3];
#pragma unroll
    for (int k = 0; k < 8; k++) acc[k & 3] += t[k] * b[j + k];
  }
  for (; j < j1; j++) acc[0] += col[(size_t)j * n3] * b[j];
  part[w][lane] = (acc[0] + acc[1]) + (acc[2] + acc[3]);
  __syncthreads();
  if (w == 0 && i < n3) {
    double t = 0.0;
#pragma unroll
    for (int k = 0; k < kRedApplyWaves; k++) t += part[k][lane];
    x[3 * (size_t)a.tgt_out[tb + i / 3] + i % 3] = t;
  }
}

// Many blocks, bound by their bytes: a thread per row, its columns in order;
// long runs of rows, 2 KB of a column at a time, read memory best.
constexpr int kRedRowThreads = 256;
__global__ __launch_bounds__(kRedRowThreads) void k_red_apply_row(RedArgs a, const double *__restrict__ v,
                                                                  double *__restrict__ x) {
  extern __shared__ double b[];
  const int li = blockIdx.x;
  const int n = a.leaves[li];
  const int tb = a.tgt_ptr[n], n3 = 3 * (a.tgt_ptr[n + 1] - tb);
  const int i0 = blockIdx.y * kRedRowThreads;
  if (i0 >= n3) return;  // the whole workgroup
  const double *Inv = a.blk + a.off[li];
  for (int i = threadIdx.x; i < n3; i += kRedRowThreads) b[i] = v[3 * (size_t)a.tgt_out[tb + i / 3] + i % 3];
  __syncthreads();
  const int i = i0 + threadIdx.x;
  if (i < n3) {
    double acc = 0.0;
    for (int j = 0; j < n3; j++) acc += Inv[(size_t)j * n3 + i] * b[j];
    x[3 * (size_t)a.tgt_out[tb + i / 3] + i % 3] = acc;
  }
}

// Small blocks: a leaf of at most T rows per workgroup; T / n3 threads share a
// row's columns (rows fastest), their sums added in order.
template <int T>
__global__ __launch_bounds__(T) void k_red_apply_leaf(RedArgs a, const double *__restrict__ v, double *__restrict__ x) {
  __shared__ double b[T], part[T];
  const int li = blockIdx.x, tid = threadIdx.x;
  const int n = a.leaves[li];
  const int tb = a.tgt_ptr[n], n3 = 3 * (a.tgt_ptr[n + 1] - tb);
  const double *Inv = a.blk + a.off[li];
  if (tid < n3) b[tid] = v[3 * (size_t)a.tgt_out[tb + tid / 3] + tid % 3];
  __syncthreads();
  const int ns = min(T / n3, 8), sh = tid / n3, i = tid - sh * n3;
  double acc[2] = {0, 0};
  if (sh < ns) {
    const int j1 = n3 * (sh + 1) / ns;
    const double *col = Inv + i;
    int j = n3 * sh / ns;
    for (; j + 8 <= j1; j += 8) {
      double t[8];
#pragma unroll
      for (int k = 0; k < 8; k++) t[k] = col[(size_t)(j + k) * n3];
#pragma unroll
      for (int k = 0; k < 8; k++) acc[k & 1] += t[k] * b[j + k];
    }
    for (; j < j1; j++) acc[0] += col[(size_t)j * n3] * b[j];
  }
  part[tid] = acc[0] + acc[1];
  __syncthreads();
  if (tid < n3) {
    double t = part[tid];
    for (int k = 1; k < ns; k++) t += part[k * n3 + tid];
    x[3 * (size_t)a.tgt_out[tb + tid / 3] + tid % 3] = t;
  }
}

void Fmm::reduced_factor() {
  const Tree &T = tree_;
  if (T.npot != T.ntgt || T.npts != T.npot)
    throw Error(NNK_EARG, "reducedSolve needs potential points == target points");
  std::vector<int32_t> tl(n_tleaves_), tp(T.count + 2);
  NNK_HIP(hipMemcpy(tl.data(), tleaves_.p, sizeof(int32_t) * n_tleaves_, hipMemcpyDeviceToHost));
  NNK_HIP(hipMemcpy(tp.data(), tgt_ptr_.p, sizeof(int32_t) * (T.count + 2), hipMemcpyDeviceToHost));
  // first entry of each leaf's block, its rows, and its diagonal tiles' inverses
  std::vector<int64_t> off(n_tleaves_ + 1, 0), poff(n_tleaves_ + 1, 0), doff(n_tleaves_ + 1, 0);
  red_maxn_ = 0;
  for (int i = 0; i < n_tleaves_; i++) {
    int64_t n3 = 3 * (tp[tl[i] + 1] - tp[tl[i]]);
    off[i + 1] = off[i] + n3 * n3;
    poff[i + 1] = poff[i] + n3;
    doff[i + 1] = doff[i] + (n3 + kInvB - 1) / kInvB * 2 * kInvB * kInvB;
    red_maxn_ = std::max<int>(red_maxn_, (int)n3);
  }
  if ((size_t)red_maxn_ * sizeof(double) > 64 * 1024)
    throw Error(NNK_ESTATE, "reducedSolve: leaf block larger than 8192 unknowns");
  std::vector<int32_t> o2l(T.ntgt, 0);
  {
    std::vector<int32_t> to(T.ntgt);
    NNK_HIP(hipMemcpy(to.data(), tgt_out_.p, sizeof(int32_t) * T.ntgt, hipMemcpyDeviceToHost));
    for (int i = 0; i < n_tleaves_; i++)
      for (int k = tp[tl[i]]; k < tp[tl[i] + 1]; k++) o2l[to[k]] = k - tp[tl[i]];
  }
  red_off_.upload(off);
  DBuf dpoff;   // poff, then doff
  const int64_t *const ddoff = [&] {
    std::vector<int64_t> both = poff;
    both.insert(both.end(), doff.begin(), doff.end());
    dpoff.upload(both);
    return dpoff.as<int64_t>() + poff.size();
  }();
  red_ord2loc_.upload(o2l);
  red_blk_.alloc(sizeof(double) * (off.back() + doff.back()));   // the tiles' inverses behind the blocks
  red_piv_.alloc(sizeof(int32_t) * std::max<int64_t>(poff.back(), 1));
  red_perm_.alloc(sizeof(int32_t) * std::max<int64_t>(poff.back(), 1));
  red_poff_ = std::move(dpoff);
  RedArgs a = red_args();
  if (n_tleaves_) {
    hipLaunchKernelGGL(k_red_form, dim3(n_tleaves_), dim3(256), 0, 0, a);
    NNK_HIP(hipGetLastError());
    for (int k0 = 0; k0 < red_maxn_; k0 += kLuNB) {
      const int left = red_maxn_ - k0;
      if (left > kLuRows) {
        hipLaunchKernelGGL(k_red_lu_panel_mem, dim3(n_tleaves_), dim3(kLuThreads), 0, 0, a, k0);
      } else {
        if (left > 512) hipLaunchKernelGGL(k_red_lu_panel<1024>, dim3(n_tleaves_), dim3(1024), 0, 0, a, k0);
        else if (left > 256) hipLaunchKernelGGL(k_red_lu_panel<512>, dim3(n_tleaves_), dim3(512), 0, 0, a, k0);
        else hipLaunchKernelGGL(k_red_lu_panel<256>, dim3(n_tleaves_), dim3(256), 0, 0, a, k0);
        hipLaunchKernelGGL(k_red_lu_rows, dim3(n_tleaves_, (red_maxn_ + 255) / 256), dim3(256), 0, 0, a, k0);
      }
      const int m = red_maxn_ - k0 - kLuNB;
      if (m > 0) {
        const int nt = (m + kLuT - 1) / kLuT;
        hipLaunchKernelGGL(k_red_lu_update, dim3(n_tleaves_, nt * nt), dim3(256), 0, 0, a, k0);
      }
    }
    NNK_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_red_perm, dim3((n_tleaves_ + 63) / 64), dim3(64), 0, 0, a, n_tleaves_);
    NNK_HIP(hipGetLastError());
    // the blocks' inverses replace their factors: each solve is then one
    // pass over them at HBM bandwidth instead of a chain of substitutions
    DBuf W;
    double *D = red_blk_.as<double>() + off.back();
    W.alloc(sizeof(double) * std::max<int64_t>(off.back(), 1));
    hipLaunchKernelGGL(k_red_diag, dim3(n_tleaves_, (red_maxn_ + kInvB - 1) / kInvB), dim3(64), 0, 0, a,
                       ddoff, D);
    hipLaunchKernelGGL(k_red_inv, dim3(n_tleaves_, (red_maxn_ + 63) / 64), dim3(256), 0, 0, a, ddoff, D,
                       W.as<double>());
    NNK_HIP(hipGetLastError());
    NNK_HIP(hipDeviceSynchronize());
    red_blk_ = std::move(W);
  }
  red_piv_ = DBuf();
  red_perm_ = DBuf();
  NNK_HIP(hipDeviceSynchronize());
  red_ready_ = true;
}

RedArgs Fmm::red_args() const {
  RedArgs a{};
  a.leaves = tleaves_.as<int32_t>();
  a.tgt_ptr = tgt_ptr_.as<int32_t>();
  a.tgt_pos = tgt_pos_.as<double>();
  a.tgt_out = tgt_out_.as<int32_t>();
  a.src_ptr = src_ptr_.as<int32_t>();
  a.src_pos = src_pos_.as<double>();
  a.ctr_ptr = ctr_ptr_.as<int64_t>();
  a.ctr_col = ctr_col_.as<int32_t>();
  a.ctr_w = ctr_w_.as<double>();
  a.ord2loc = red_ord2loc_.as<int32_t>();
  a.off = red_off_.as<int64_t>();
  a.blk = red_blk_.as<double>();
  a.piv = red_piv_.as<int32_t>();
  a.perm = red_perm_.as<int32_t>();
  a.poff = red_poff_.as<int64_t>();
  a.e2 = eps_ * eps_;
  a.c = 1.0 / (8.0 * kPi * mu_);
  a.nearest = tree_.nearest ? 1 : 0;
  return a;
}

void Fmm::reduced_solve(const double *d_v, double *d_f, hipStream_t s) {
  if (!red_ready_) reduced_factor();
  if (!n_tleaves_) return;
  RedArgs a = red_args();
  auto go = [&](auto kern, int rows, int threads, size_t lds) {
    hipLaunchKernelGGL(kern, dim3(n_tleaves_, (red_maxn_ + rows - 1) / rows), dim3(threads), lds, s, a, d_v, d_f);
  };
  // Measured by number of leaves x rows per leaf (eight wavefronts per 64
  // rows; a thread per row; a leaf per workgroup), us: 32,768 x 30 113, 78, 74;
  // 32,768 x 72 412, 297, 282; 4,096 x 120 96, 89, 87; 64 x 255 13.3, 18, 13.4;
  // 512 x 234 (at most 312) 47, 39, 39; 4,096 x 220 (312) 385, 320, 319;
  // 512 x 352 (432) 107, 100, 117; 512 x 495 186, 167, 180; 64 x 330 14, 31, 22;
  // 1,807 x 166 (600) 186, 193; 512 x 586 (723) 283, 317; and by the inverses'
  // bytes: 64 x 1,500 (1.2 GB) 199, 252; 256 x 1,020 (2.1 GB) 403, 367;
  // 64 x 2,100 (2.3 GB) 400, 381; 512 x 1,500 (9.2 GB) 1,827, 1,585.
  const size_t lds = sizeof(double) * red_maxn_;
  const bool many = n_tleaves_ >= ncu_;
  // (346 x 63 (192), 11 MB, alone on the device 9.1, 27, 12.1)
  if (n_tleaves_ < 4 * ncu_ && red_blk_.bytes < ((size_t)64 << 20)) go(k_red_apply, 64, 64 * kRedApplyWaves, lds);
  else if (red_maxn_ <= 64) go(k_red_apply_leaf<128>, 64, 128, 0);
  else if (red_maxn_ <= 128) go(k_red_apply_leaf<256>, 128, 256, 0);
  else if (red_maxn_ <= 256 || (red_maxn_ <= 320 && many)) go(k_red_apply_leaf<512>, 320, 512, 0);
  else if ((red_maxn_ <= 512 && many) || red_blk_.bytes >= ((size_t)7 << 28))
    go(k_red_apply_row, kRedRowThreads, kRedRowThreads, lds);
  else go(k_red_apply, 64, 64 * kRedApplyWaves, lds);
  NNK_HIP(hipGetLastError());
}

}  // namespace nnk
