// Gathered-column block GEMM on the FP64 matrix cores (v_mfma_f64_16x16x4_f64):
//
//   C[:, cidx[n]] (+)= sum_b A_b X[:, gidx[b][n]]
//
// A_b are (3Nq x 3Nq) operators stored k-major (At[k][m], Kpad x Mpad, zero
// padded); X and C hold one density vector of length K per node.
// k_gemm_gather serves the dense M2L (189 translation operators per child
// class) and the truncated forms; k_gemm_direct below the FP64 form's M2M (8
// child operators), L2L and two-factor check-to-equivalent solves.
//
// Work decomposition: the flattened grid is walked job-fastest, so with the
// hardware's round-robin dispatch of workgroups to the 8 XCDs the 8 M2L jobs
// (one per child class) each stay on one XCD and stream their operators
// through that XCD's L2.  A workgroup owns a BM x BN tile of C; its 4 waves
// form a 2x2 grid of (BM/2) x (BN/2) sub-tiles.  K is walked in BK-deep
// chunks over the operator blocks that have at least one source in the tile,
// through a two-stage LDS ping-pong fed by register prefetch (one barrier per
// chunk).  With nsplit > 1 the active blocks are divided over nsplit
// workgroups (split-K, for levels with few tiles); each writes its partial
// tile to P[(split, job, column)] and a fixed-order reduction forms C.
// MFMA operand layout (measured on gfx950): lane l holds A[l%16][l/16]
// and B[l/16][l%16]; accumulator register r of lane l holds D[l/16 + 4r][l%16].
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "nnk_fmm.hpp"

namespace nnk {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef double d2v __attribute__((ext_vector_type(2)));
// pointers read out of a job: global, not flat, loads
typedef const double __attribute__((address_space(1))) *gcd;
typedef const int32_t __attribute__((address_space(1))) *gci;

// TAG only separates launches by role in profiles (1 = M2L translations).
template <int BM, int BN, int BK, int TAG>
__global__ __launch_bounds__(256, 2) void k_gemm_gather(int M, int K, int Mpad, int Kpad,
                                                        const double *__restrict__ X, int ldx,
                                                        double *__restrict__ C, int ldc, int beta,
                                                        const GemmJob *__restrict__ jobs,
                                                        int njobs, int nrb, int nsplit,
                                                        double *__restrict__ P, int maxN) {
  static_assert(BK == 16 && BM % 32 == 0 && BN % 32 == 0, "tile shape");
  constexpr int WM = BM / 2, WN = BN / 2, TM = WM / 16, TN = WN / 16;
  constexpr int A2 = BK * BM / 2;       // double2 per A chunk
  constexpr int B2 = BN * BK / 2;       // double2 per B chunk
  constexpr int AR = A2 / 256, BR = B2 / 256;
  static_assert(A2 % 256 == 0 && B2 % 256 == 0, "chunk must split evenly over 256 threads");
  constexpr int BKP = BK + 2;           // padded B row (keeps 16-byte alignment)
  __shared__ __attribute__((aligned(16))) double As[2][BK][BM];
  __shared__ __attribute__((aligned(16))) double Bs[2][BN][BKP];
  __shared__ int act[kMaxBlocks];
  __shared__ int nact_s;

  const int bid = blockIdx.x;
  const int jb = bid % njobs;
  int rr = bid / njobs;
  const int sp = rr % nsplit;
  rr /= nsplit;
  const int rb = rr % nrb, ct = rr / nrb;
  const GemmJob J = jobs[jb];
  const int col0 = ct * BN;
  if (col0 >= J.N) return;
  const int m0 = rb * BM;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int lr = lane & 15, lk = lane >> 4;

  // ---- operator blocks with at least one source column in this tile ----
  int nact;
  if (J.tptr) {  // precomputed per tile
    const int t0 = J.tptr[ct];
    nact = J.tptr[ct + 1] - t0;
    for (int i = tid; i < nact; i += 256) act[i] = J.tlist[t0 + i];
    __syncthreads();
  } else {
    if (tid == 0) nact_s = 0;
    __syncthreads();
    for (int b = tid; b < J.nb; b += 256) {
      bool any = false;
      if (J.gidx) {
        const int32_t *g = J.gidx + (size_t)b * J.N;
        for (int n = 0; n < BN && !any; n++)
          if (col0 + n < J.N && g[col0 + n] >= 0) any = true;
      } else {
        any = true;
      }
      if (any) {
        int slot = atomicAdd(&nact_s, 1);
        act[slot] = b;
      }
    }
    __syncthreads();
    nact = nact_s;
    // keep the walk in block order (deterministic summation order); only
    // small jobs come here (at most 8 blocks)
    if (tid == 0) {
      for (int i = 1; i < nact; i++) {
        int v = act[i], j = i - 1;
        while (j >= 0 && act[j] > v) { act[j + 1] = act[j]; j--; }
        act[j + 1] = v;
      }
    }
    __syncthreads();
  }

  d4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++) acc[i][j] = d4{0, 0, 0, 0};

  const int KC = Kpad / BK;
  const int a0 = (int)((int64_t)nact * sp / nsplit), a1 = (int)((int64_t)nact * (sp + 1) / nsplit);
  const int total = (a1 - a0) * KC;
  d2v ra[AR], rbv[BR];
  int gcol[BR];
  int cur_block = -1;

  auto fetch = [&](int c) {
    const int q = c / KC, kc = c - q * KC;
    const int b = act[a0 + q];
    const int k0 = kc * BK;
    if (b != cur_block) {
      cur_block = b;
#pragma unroll
      for (int r = 0; r < BR; r++) {
        const int i = tid + 256 * r;
        const int n = i / (BK / 2);
        const int col = col0 + n;
        int g = -1;
        if (col < J.N) g = J.gidx ? J.gidx[(size_t)b * J.N + col] : col;
        gcol[r] = g;
      }
    }
    const double *__restrict__ Ab = J.A[b];
#pragma unroll
    for (int r = 0; r < AR; r++) {
      const int i = tid + 256 * r;
      const int kk = i / (BM / 2), m2 = i - kk * (BM / 2);
      ra[r] = *reinterpret_cast<const d2v *>(Ab + (size_t)(k0 + kk) * Mpad + m0 + 2 * m2);
    }
#pragma unroll
    for (int r = 0; r < BR; r++) {
      const int i = tid + 256 * r;
      const int kk2 = i % (BK / 2);
      const int k = k0 + 2 * kk2;
      d2v v = {0.0, 0.0};
      if (gcol[r] >= 0) {
        const double *xp = X + (size_t)gcol[r] * ldx + k;
        if (k + 1 < K) v = d2v{xp[0], xp[1]};
        else if (k < K) v = d2v{xp[0], 0.0};
      }
      rbv[r] = v;
    }
  };
  auto stash = [&](int buf) {
#pragma unroll
    for (int r = 0; r < AR; r++) {
      const int i = tid + 256 * r;
      const int kk = i / (BM / 2), m2 = i - kk * (BM / 2);
      *reinterpret_cast<d2v *>(&As[buf][kk][2 * m2]) = ra[r];
    }
#pragma unroll
    for (int r = 0; r < BR; r++) {
      const int i = tid + 256 * r;
      const int n = i / (BK / 2), kk2 = i % (BK / 2);
      *reinterpret_cast<d2v *>(&Bs[buf][n][2 * kk2]) = rbv[r];
    }
  };

  if (total > 0) {
    fetch(0);
    stash(0);
    __syncthreads();
    for (int c = 0; c < total; c++) {
      const int buf = c & 1;
      if (c + 1 < total) fetch(c + 1);
#pragma unroll
      for (int ks = 0; ks < BK; ks += 4) {
        double av[TM], bv[TN];
#pragma unroll
        for (int i = 0; i < TM; i++) av[i] = As[buf][ks + lk][wm * WM + i * 16 + lr];
#pragma unroll
        for (int j = 0; j < TN; j++) bv[j] = Bs[buf][wn * WN + j * 16 + lr][ks + lk];
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
          for (int j = 0; j < TN; j++)
            acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[i], bv[j], acc[i][j], 0, 0, 0);
      }
      if (c + 1 < total) stash(buf ^ 1);
      __syncthreads();
    }
  }
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++) {
      const int col = col0 + wn * WN + j * 16 + lr;
      if (col >= J.N) continue;
      const int cs = J.cidx ? J.cidx[col] : col;
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int row = m0 + wm * WM + i * 16 + lk + 4 * r;
        if (row >= M) continue;
        if (nsplit > 1) {
          P[((size_t)(sp * njobs + jb) * maxN + col) * ldc + row] = acc[i][j][r];
        } else {
          double *p = C + (size_t)cs * ldc + row;
          *p = beta ? *p + acc[i][j][r] : acc[i][j][r];
        }
      }
    }
}

// The same product for the FP64 form's M2M, L2L and check-to-equivalent
// solves (jobs of one or eight operator blocks), without LDS staging.  An FP64
// MFMA holds the matrix core for 64 cycles, so a wavefront of TM x TN tiles of
// 16 x 16 needs one fragment load per TM TN / (TM + TN) products: little
// enough to load the fragments straight from memory, one 16-deep K chunk
// ahead, with no barrier to wait at.  Within a chunk lane group lk = lane / 16
// takes k = 4 lk .. 4 lk + 3 (32 contiguous bytes of a column); product s
// takes the s-th of each group.  KS = 1: the four wavefronts of a workgroup
// take the same rows of neighbouring column tiles (three of them read A from
// L1).  KS > 1: KS wavefronts share one tile and split its (block, chunk)
// sequence, their sums added in wavefront order through LDS: for launches of
// few tiles, which are bound by the latency of the chunks in a row.
// The row blocks of a column tile are 8 workgroups apart, on one XCD, so its
// columns come from one L2.
// ORD (KS = 1): the summation order of k_gemm_gather, to the bit: product s of a
// chunk takes k = 4 s + lk.
template <int TM, int TN, int KS, bool ORD = false>
__global__ __launch_bounds__(KS > 4 ? 64 * KS : 256, 2) void k_gemm_direct(
    int M, int K, int Mpad, int Kpad, const double *__restrict__ X, int ldx, double *__restrict__ C, int ldc, int beta,
    const GemmJob *__restrict__ jobs, int njobs, int nrb, int nct) {
  static_assert(!ORD || KS == 1, "one chain per sum");
  constexpr int WAVES = KS > 4 ? KS : 4, CW = WAVES / KS;   // wavefronts, column tiles of a workgroup
  __shared__ double red[KS > 1 ? (WAVES - CW) * TM * TN * 256 : 1];
  __shared__ int act[kMaxBlocks], nact_s;
  const int q = blockIdx.x >> 3, u = (q / nrb) * 8 + (blockIdx.x & 7), rb = q % nrb;
  if (u >= njobs * nct) return;
  const GemmJob J = jobs[u % njobs];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lk = lane >> 4;
  const int ks = wave / CW, wc = wave % CW;
  const int wg0 = (u / njobs) * CW * TN * 16;    // first column of the workgroup
  if (wg0 >= J.N) return;
  // operator blocks with a source in the workgroup's columns, in order
  if (wave == 0) {
    int n = 0;
    for (int b = 0; b < J.nb; b++) {
      bool any = true;
      if (J.gidx) {
        any = false;
        for (int c = lane; c < CW * TN * 16; c += 64) any |= wg0 + c < J.N && ((gci)J.gidx)[(size_t)b * J.N + wg0 + c] >= 0;
        any = __ballot(any) != 0;
      }
      if (any) {
        if (lane == 0) act[n] = b;
        n++;
      }
    }
    if (lane == 0) nact_s = n;
  }
  __syncthreads();
  const int KC = Kpad / 16, total = nact_s * KC;
  const int col0 = wg0 + wc * TN * 16;
  const int rt0 = rb * TM;                       // first row tile; past the last: its rows are not stored
  d4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++) acc[i][j] = d4{0, 0, 0, 0};
  int cur = -1;
  gcd Ab = nullptr;
  gcd xc[TN];
  bool on[TN];
  // Branch-free: a lane without a source loads node 0's values and a lane past
  // the columns' end the last four; lo is the first product that counts.
  auto fetch = [&](int c, double (&a)[4][TM], double (&x)[TN][4], int (&lo)[TN]) {
    const int qb = c / KC, k0 = (c - qb * KC) * 16 + 4 * lk;
    if (qb != cur) {
      cur = qb;
      const int b = act[qb];
      Ab = (gcd)((const uint64_t __attribute__((address_space(1))) *)J.A)[b];
#pragma unroll
      for (int j = 0; j < TN; j++) {
        const int col = col0 + j * 16 + lr;
        int g = -1;
        if (col < J.N) g = J.gidx ? ((gci)J.gidx)[(size_t)b * J.N + col] : col;
        on[j] = g >= 0;
        xc[j] = (gcd)X + (size_t)(g < 0 ? 0 : g) * ldx;
      }
    }
    if constexpr (ORD) {
#pragma unroll
      for (int s = 0; s < 4; s++) {
        const int k = min(k0 - 3 * lk + 4 * s, K - 1);   // (chunk start) + lk + 4 s
#pragma unroll
        for (int i = 0; i < TM; i++) a[s][i] = Ab[(size_t)k * Mpad + min((rt0 + i) * 16, Mpad - 16) + lr];
#pragma unroll
        for (int j = 0; j < TN; j++) x[j][s] = xc[j][k];
      }
      // hi: products with k < K count
#pragma unroll
      for (int j = 0; j < TN; j++) lo[j] = on[j] ? (K - (k0 - 3 * lk) + 3) / 4 : 0;
      return;
    }
    const int kb = max(min(k0, K - 4), 0);
#pragma unroll
    for (int s = 0; s < 4; s++)
#pragma unroll
      for (int i = 0; i < TM; i++) a[s][i] = Ab[(size_t)(kb + s) * Mpad + min((rt0 + i) * 16, Mpad - 16) + lr];
#pragma unroll
    for (int j = 0; j < TN; j++) {
#pragma unroll
      for (int s = 0; s < 4; s++) x[j][s] = xc[j][kb + s];
      lo[j] = on[j] ? k0 - kb : 4;
    }
  };
  auto product = [&](const double (&a)[4][TM], const double (&x)[TN][4], const int (&lo)[TN]) {
#pragma unroll
    for (int s = 0; s < 4; s++) {
      double v[TN];
#pragma unroll
      for (int j = 0; j < TN; j++) v[j] = (ORD ? s < lo[j] : s >= lo[j] && s < K) ? x[j][s] : 0.0;
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[s][i], v[j], acc[i][j], 0, 0, 0);
    }
  };
  double a0[4][TM], a1[4][TM], x0[TN][4], x1[TN][4];
  int l0[TN], l1[TN];
  // the wavefront's chunks: a contiguous share of the sequence, in pairs; a
  // chunk past the end counts for nothing
  const int c0 = (int)((int64_t)total * ks / KS), c1 = (int)((int64_t)total * (ks + 1) / KS);
  if (c0 < c1) {
    fetch(c0, a0, x0, l0);
#pragma unroll 1
    for (int c = c0; c < c1; c += 2) {
      fetch(min(c + 1, c1 - 1), a1, x1, l1);
      if (c + 1 == c1)
#pragma unroll
        for (int j = 0; j < TN; j++) l1[j] = ORD ? 0 : 4;
      __builtin_amdgcn_sched_barrier(0);   // the loads go out before the products, not among them
      product(a0, x0, l0);
      fetch(min(c + 2, c1 - 1), a0, x0, l0);
      __builtin_amdgcn_sched_barrier(0);
      product(a1, x1, l1);
    }
  }
  if constexpr (KS > 1) {
    auto slot = [&](int k, int e) { return ((((k - 1) * CW + wc) * TM * TN * 4) + e) * 64 + lane; };
    if (ks > 0)
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
          for (int r = 0; r < 4; r++) red[slot(ks, (i * TN + j) * 4 + r)] = acc[i][j][r];
    __syncthreads();
    if (ks > 0) return;
    for (int k = 1; k < KS; k++)
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
          for (int r = 0; r < 4; r++) acc[i][j][r] += red[slot(k, (i * TN + j) * 4 + r)];
  }
#pragma unroll
  for (int j = 0; j < TN; j++) {
    const int col = col0 + j * 16 + lr;
    if (col >= J.N) continue;
    double *p = C + (size_t)(J.cidx ? J.cidx[col] : col) * ldc;
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int row = (rt0 + i) * 16 + lk + 4 * r;
        if (row < M) p[row] = beta ? p[row] + acc[i][j][r] : acc[i][j][r];
      }
  }
}

// Launches the product by its number of workgroups: one wavefront per tile
// (48 x 128 per workgroup) from two workgroups per CU, 48 x 32 shared by four
// wavefronts from one per CU, else 32 x 16 shared by eight.  Both sides of the
// lines at K = 456: 4,096 columns (320 workgroups of 48 x 128) take 0.16 ms
// less over a matvec's up pass with the shared tiles; 512 columns 36 against
// 23 us for an L2L.  Other ranks, a matvec's up pass in us by the rule and with
// each shape throughout (48 x 128; 48 x 32; 32 x 16): K = 168, 512 leaves 43
// (165; 70; 42), 4,096 leaves 88 (299; 129; 106), 32,768 leaves 257 (522; 365;
// 550); K = 888, 512 leaves 166 (696; 234; 184), 8,192 leaves 1,120 (2,221;
// 1,272; 1,850); K = 1,464, 512 leaves 388 (1,131; 371; 464), 2,048 leaves 1,089
// (2,224; 922; 1,358): at the largest rank the shared tiles would be the better a
// little earlier.
// FP64 matvecs before (160 x 32 tiles staged through LDS, M2M split over the
// children where columns are few) and now, res 6: up pass 198 -> 76 us, solves
// 155 -> 46 us, L2L 49 -> 23 us with 64 and 512 leaves; 2^20 points 1.42 ->
// 1.11 ms, 0.91 -> 0.71 ms, 0.46 -> 0.40 ms.
inline void launch_gemm_direct(int M, int K, int Mpad, int Kpad, const double *X, int ldx, double *C, int ldc,
                               int beta, const GemmJob *jobs, int njobs, int maxN, hipStream_t s) {
  auto wgs = [&](int rows, int cols) {
    return (int64_t)njobs * ((M + rows - 1) / rows) * ((maxN + cols - 1) / cols);
  };
  auto go = [&](auto kern, int threads, int rows, int cols) {
    const int nrb = (M + rows - 1) / rows, nct = (maxN + cols - 1) / cols;
    const int64_t units = ((int64_t)njobs * nct + 7) / 8 * 8;
    hipLaunchKernelGGL(kern, dim3((unsigned)(units * nrb)), dim3(threads), 0, s, M, K, Mpad, Kpad, X, ldx, C, ldc,
                       beta, jobs, njobs, nrb, nct);
    NNK_HIP(hipGetLastError());
  };
  if (wgs(48, 128) >= 512) go(k_gemm_direct<3, 2, 1>, 256, 48, 128);
  else if (wgs(48, 32) >= 256) go(k_gemm_direct<3, 2, 4>, 256, 48, 32);
  else go(k_gemm_direct<2, 1, 8>, 512, 32, 16);
}

// The product in k_gemm_gather's order, for the truncated forms' launches of few
// of its tiles.  False: not launched, k_gemm_gather is the faster.  L2L of a
// 20-body suspension (up to 144 tiles per level) 0.215 -> 0.137 ms; of 10^5
// clustered points, levels of 192 to 512 tiles included, 0.45 against 0.52 ms.
inline bool launch_gemm_ordered(int M, int K, int Mpad, int Kpad, const double *X, int ldx, double *C, int ldc,
                                int beta, const GemmJob *jobs, int njobs, int maxN, hipStream_t s) {
  if ((int64_t)njobs * (Mpad / GBM) * ((maxN + GBN0 - 1) / GBN0) >= 192) return false;
  const int nrb = (M + 31) / 32, nct = (maxN + 63) / 64;
  const int64_t units = ((int64_t)njobs * nct + 7) / 8 * 8;
  hipLaunchKernelGGL((k_gemm_direct<2, 1, 1, true>), dim3((unsigned)(units * nrb)), dim3(256), 0, s, M, K, Mpad, Kpad, X,
                     ldx, C, ldc, beta, jobs, njobs, nrb, nct);
  NNK_HIP(hipGetLastError());
  return true;
}

// C[slot[c]][row] = sum over splits of P[split][c][row], splits in order
// (c runs over job * maxN + column; slot -1 = no column)
__global__ void k_split_reduce(const int32_t *__restrict__ slot, int M, int ldc, int nsplit,
                               const double *__restrict__ P, size_t pstride, double *__restrict__ C);

}  // namespace nnk
