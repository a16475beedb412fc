// M2L of the FP64 forms in frequency space.
//
// The up surface of a box is a res^3 grid without its interior, and the
// check potentials of a V-list pair are evaluated on the same grid of the
// target box, so a translation is a 3-D convolution: with grid spacing h,
// box width w and source offset o, chk[t] = sum_s k_o[t - s] u[s] with
// k_o[d] = S(d h - o w).  On n = 2 res - 1 points per axis (the differences
// -(res-1) .. res-1, no padding beyond them) the discrete Fourier transform
// turns it into one 3 x 3 complex product per frequency.  n is odd, so
// (n^3 + 1) / 2 frequencies determine the real transform.
//
// The V list of a box is the children of its parent's 26 neighbours that
// are not adjacent to it, so per frequency and neighbour direction the
// interactions of the 8 children of a parent with the 8 children of the
// neighbour are one 24 x 24 complex block (adjacent pairs: zero operators),
// shared by every parent of the level: an FP64 MFMA product with 48 real
// rows, 26 x 48 real columns and one column per target parent.  At res 6 a
// full neighbourhood costs 666 x 26 x 4608 flop = 80 Mflop per parent
// against 629 Mflop for the 8 x 189 dense 456 x 456 translations.
//
// Measured at 2^20 uniform points, 64 per leaf, res 6 (4,681 parents): M2L
// 56.5 -> 6.5 ms (products 5.9 ms at 62 TF/s of the 78.6 TF/s FP64 matrix
// peak, transforms 0.3 ms each way at ~4 TB/s), matvec 61.2 -> 11.0 ms; at
// 3,000 points (72 parents) 1.0 -> 0.18 ms; on a 64-spheroid suspension,
// whose parents have few of the 26 neighbours and children, 2.8 -> 2.1 ms.
#include <algorithm>
#include <array>
#include <cmath>
#include <cstdlib>

#include "nnk_fmm.hpp"
#include "nnk_kernels.hpp"
#include "nnk_spectral.hpp"

namespace nnk {

namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef double d2v __attribute__((ext_vector_type(2)));

// Frequencies (kx, ky, kz) with kx = 0 .. res-1; the kx = 0 plane keeps
// (0, 0 .. res-1) and (1 .. res-1, all kz), the other half of it being
// complex conjugates.
__host__ __device__ constexpr int plane_base(int P, int kx) {
  const int n = 2 * P - 1;
  return kx == 0 ? 0 : P + (P - 1) * n + (kx - 1) * n * n;
}
template <int P> __device__ __forceinline__ int freq_index(int kx, int ky, int kz) {
  constexpr int n = 2 * P - 1;
  if (kx == 0) return ky == 0 ? kz : P + (ky - 1) * n + kz;
  return plane_base(P, kx) + ky * n + kz;
}

// the 13th of the 27 directions is the parent itself
__host__ __device__ constexpr int dir27(int d) { return d + (d >= 13); }

// Operator table of one level, one workgroup per (offset slot, component):
// the kernel on the n^3 differences, then the transform axis by axis, one
// kx plane at a time.  Set-up only.
template <int P>
__global__ __launch_bounds__(256) void k_spec_table(double w, double e2, double c, const double *__restrict__ tw,
                                                    double *__restrict__ tab) {
  constexpr int n = 2 * P - 1;
  __shared__ double g[n * n * n];
  __shared__ d2v a[n * n], b[n * n];
  __shared__ d2v tws[n];
  const int sl = blockIdx.x, comp = blockIdx.y, tid = threadIdx.x;
  const int ox = sl / 49 - 3, oy = (sl / 7) % 7 - 3, oz = sl % 7 - 3;
  if (max(abs(ox), max(abs(oy), abs(oz))) < 2) return;   // adjacent: stays zero
  const int ci = comp < 3 ? 0 : comp < 5 ? 1 : 2, cj = comp < 3 ? comp : comp < 5 ? comp - 2 : 2;
  const double h = w / (P - 1);
  for (int i = tid; i < n; i += 256) tws[i] = d2v{tw[2 * i], tw[2 * i + 1]};
  for (int i = tid; i < n * n * n; i += 256) {
    const int z = i % n, y = (i / n) % n, x = i / (n * n);
    const double r[3] = {(x < P ? x : x - n) * h - ox * w, (y < P ? y : y - n) * h - oy * w,
                         (z < P ? z : z - n) * h - oz * w};
    const double r2 = r[0] * r[0] + r[1] * r[1] + r[2] * r[2];
    const double inv = rsqrt(r2 + e2);
    g[i] = (r[ci] * r[cj] + (ci == cj ? r2 + 2.0 * e2 : 0.0)) * (c * inv * inv * inv);
  }
  __syncthreads();
  const double norm = 2.0 / ((double)n * n * n);
  for (int kx = 0; kx < P; kx++) {
    for (int i = tid; i < n * n; i += 256) {
      double re = 0, im = 0;
      for (int x = 0; x < n; x++) {
        const d2v t = tws[(kx * x) % n];
        const double v = g[x * n * n + i];
        re += v * t[0];
        im -= v * t[1];
      }
      a[i] = d2v{re, im};
    }
    __syncthreads();
    for (int i = tid; i < n * n; i += 256) {
      const int ky = i / n, z = i % n;
      double re = 0, im = 0;
      for (int y = 0; y < n; y++) {
        const d2v t = tws[(ky * y) % n], v = a[y * n + z];
        re += v[0] * t[0] + v[1] * t[1];
        im += v[1] * t[0] - v[0] * t[1];
      }
      b[i] = d2v{re, im};
    }
    __syncthreads();
    for (int i = tid; i < n * n; i += 256) {
      const int ky = i / n, kz = i % n;
      if (kx == 0 && (ky == 0 ? kz >= P : ky >= P)) continue;
      double re = 0, im = 0;
      for (int z = 0; z < n; z++) {
        const d2v t = tws[(kz * z) % n], v = b[ky * n + z];
        re += v[0] * t[0] + v[1] * t[1];
        im += v[1] * t[0] - v[0] * t[1];
      }
      // the inverse transform takes twice the real part of every kept
      // frequency but the constant one
      const double f = (kx | ky | kz) == 0 ? 0.5 * norm : norm;
      double *o = tab + (((size_t)freq_index<P>(kx, ky, kz) * 343 + sl) * 6 + comp) * 2;
      o[0] = f * re;
      o[1] = f * im;
    }
    __syncthreads();
  }
}

// v[k] for k = 0 .. n-1 (n = 2P-1) of the P inputs g: cosine and sine sums
// serve k and n-k at once.  tw[m] = (cos, sin)(2 pi m / n), uniform.
template <int P, class F>
__device__ __forceinline__ void dft_fwd(const d2v (&g)[P], const double *__restrict__ tw, F &&out) {
  constexpr int n = 2 * P - 1;
  {
    d2v s = g[0];
#pragma unroll
    for (int y = 1; y < P; y++) s += g[y];
    out(0, s);
  }
#pragma unroll
  for (int k = 1; k < P; k++) {
    d2v A = g[0], B = {0.0, 0.0};
#pragma unroll
    for (int y = 1; y < P; y++) {
      const double cv = tw[2 * ((k * y) % n)], sv = tw[2 * ((k * y) % n) + 1];
      A += cv * g[y];
      B += sv * g[y];
    }
    out(k, d2v{A[0] + B[1], A[1] - B[0]});       // sum g e^{-i}
    out(n - k, d2v{A[0] - B[1], A[1] + B[0]});
  }
}

// Forward transform of one source parent's 8 children: 24 fields (child,
// component).  A thread keeps its (child, component, y, z) lines along x in
// registers over all kx of the workgroup; per kx the x sums, then y, then z,
// with the intermediates in LDS, the field fastest.
// X[frequency][parent][child][component][re im]: 384 contiguous bytes per
// (frequency, parent).  Workgroup y takes kxn planes from kx0 on (few
// parents: one plane each, so that the chip fills; many: all of them, so
// that the densities are read once).
template <int P, int T>
__global__ __launch_bounds__(T) void k_spec_fwd(const double *__restrict__ up, int K, const int32_t *__restrict__ src0,
                                                const int32_t *__restrict__ smask, const int32_t *__restrict__ qmap,
                                                const double *__restrict__ tw, int kx0, int nkx, int kxn,
                                                double *__restrict__ X, size_t fstride) {
  constexpr int n = 2 * P - 1, NL = (24 * P * P + T - 1) / T;
  __shared__ d2v a[P * P * 24], b[P * n * 24];
  const int sp = blockIdx.x, tid = threadIdx.x;
  const int ka = kx0 + blockIdx.y * kxn, kb = min(ka + kxn, kx0 + nkx);
  const int c0 = src0[sp], mask = smask[sp];
  double u[NL][P];
#pragma unroll
  for (int l = 0; l < NL; l++) {
    const int i = tid + l * T;
    const int c = i % 3, y = (i / 3) % P, z = (i / (3 * P)) % P, ch = i / (3 * P * P);
    const bool on = i < 24 * P * P && ((mask >> (ch & 7)) & 1);
#pragma unroll
    for (int x = 0; x < P; x++) {
      const int q = on ? qmap[(x * P + z) * P + y] : -1;
      u[l][x] = q >= 0 ? up[(size_t)(c0 + ch) * K + 3 * q + c] : 0.0;
    }
  }
  const int fb = plane_base(P, kx0);
  for (int kx = ka; kx < kb; kx++) {
#pragma unroll
    for (int l = 0; l < NL; l++) {
      const int i = tid + l * T;
      if (i < 24 * P * P) {
        const int c = i % 3, y = (i / 3) % P, z = (i / (3 * P)) % P, ch = i / (3 * P * P);
        double re = u[l][0], im = 0;
#pragma unroll
        for (int x = 1; x < P; x++) {
          const int m = (kx * x) % n;
          re += u[l][x] * tw[2 * m];
          im -= u[l][x] * tw[2 * m + 1];
        }
        a[(z * P + y) * 24 + ch * 3 + c] = d2v{re, im};
      }
    }
    __syncthreads();
    for (int i = tid; i < 24 * P; i += T) {
      const int f = i % 24, z = i / 24;
      d2v g[P];
#pragma unroll
      for (int y = 0; y < P; y++) g[y] = a[(z * P + y) * 24 + f];
      dft_fwd<P>(g, tw, [&](int ky, d2v v) { b[(ky * P + z) * 24 + f] = v; });
    }
    __syncthreads();
    const int kyn = kx == 0 ? P : n;
    for (int i = tid; i < 24 * kyn; i += T) {
      const int f = i % 24, ky = i / 24;
      d2v g[P];
#pragma unroll
      for (int z = 0; z < P; z++) g[z] = b[(ky * P + z) * 24 + f];
      double *o = X + (size_t)sp * 48 + 2 * f;
      const int base = freq_index<P>(kx, ky, 0) - fb;
      const bool half = kx == 0 && ky == 0;
      dft_fwd<P>(g, tw, [&](int kz, d2v v) {
        if (!half || kz < P) *reinterpret_cast<d2v *>(o + (size_t)(base + kz) * fstride) = v;
      });
    }
  }
}

// g[z] for z = 0 .. P-1 from the n frequencies in(k): sum v e^{+i}
template <int P, class F>
__device__ __forceinline__ void dft_inv(d2v (&g)[P], const double *__restrict__ tw, F &&in) {
  constexpr int n = 2 * P - 1;
  const d2v v0 = in(0);
#pragma unroll
  for (int z = 0; z < P; z++) g[z] = v0;
#pragma unroll
  for (int k = 1; k < P; k++) {
    const d2v u = in(k), v = in(n - k);
    const d2v S = u + v, D = u - v;
    g[0] += S;
#pragma unroll
    for (int z = 1; z < P; z++) {
      const double cv = tw[2 * ((k * z) % n)], sv = tw[2 * ((k * z) % n) + 1];
      g[z][0] += cv * S[0] - sv * D[1];
      g[z][1] += cv * S[1] + sv * D[0];
    }
  }
}

// Inverse transform of CG children of one target parent: z then y per kx,
// the x sums of every kx in registers, one (child, component, y, z) line
// per thread and pass.  add: check potentials accumulate (kx planes done in
// several launches).
template <int P, int CG, int T>
__global__ __launch_bounds__(T) void k_spec_inv(const double *__restrict__ Y, size_t fstride, int K,
                                                const int32_t *__restrict__ tgt0, const int32_t *__restrict__ tmask,
                                                const int32_t *__restrict__ qmap, const double *__restrict__ tw, int kx0,
                                                int nkx, int add, double *__restrict__ chk) {
  constexpr int n = 2 * P - 1, NF = 3 * CG, NL = (NF * P * P + T - 1) / T;
  __shared__ d2v b[P * n * NF], a[P * P * NF];
  const int t = blockIdx.x / (8 / CG), g0 = (blockIdx.x % (8 / CG)) * CG, tid = threadIdx.x;
  const int mask = (tmask[t] >> g0) & ((1 << CG) - 1);
  if (!mask) return;
  double acc[NL][P];
#pragma unroll
  for (int l = 0; l < NL; l++)
#pragma unroll
    for (int x = 0; x < P; x++) acc[l][x] = 0.0;
  const int fb = plane_base(P, kx0);
  const double *yp = Y + (size_t)t * 48 + 6 * g0;
  for (int kx = kx0; kx < kx0 + nkx; kx++) {
    const int kyn = kx == 0 ? P : n;
    for (int i = tid; i < NF * kyn; i += T) {
      const int f = i % NF, ky = i / NF;
      const double *o = yp + (size_t)(freq_index<P>(kx, ky, 0) - fb) * fstride + 2 * f;
      const bool half = kx == 0 && ky == 0;
      d2v g[P];
      dft_inv<P>(g, tw, [&](int kz) {
        if (half && kz >= P) return d2v{0.0, 0.0};
        return *reinterpret_cast<const d2v *>(o + (size_t)kz * fstride);
      });
#pragma unroll
      for (int z = 0; z < P; z++) b[(z * n + ky) * NF + f] = g[z];
    }
    __syncthreads();
    for (int i = tid; i < NF * P; i += T) {
      const int f = i % NF, z = i / NF;
      d2v g[P];
      dft_inv<P>(g, tw, [&](int ky) {
        if (ky >= kyn) return d2v{0.0, 0.0};
        return b[(z * n + ky) * NF + f];
      });
#pragma unroll
      for (int y = 0; y < P; y++) a[(z * P + y) * NF + f] = g[y];
    }
    __syncthreads();
#pragma unroll
    for (int l = 0; l < NL; l++) {
      const int i = tid + l * T;
      if (i < NF * P * P) {
        const int c = i % 3, y = (i / 3) % P, z = (i / (3 * P)) % P, ch = i / (3 * P * P);
        const d2v v = a[(z * P + y) * NF + ch * 3 + c];
#pragma unroll
        for (int x = 0; x < P; x++) {
          const int m = (kx * x) % n;
          acc[l][x] += v[0] * tw[2 * m] - v[1] * tw[2 * m + 1];
        }
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int l = 0; l < NL; l++) {
    const int i = tid + l * T;
    if (i >= NF * P * P) continue;
    const int c = i % 3, y = (i / 3) % P, z = (i / (3 * P)) % P, ch = i / (3 * P * P);
    if (!((mask >> ch) & 1)) continue;
    double *o = chk + (size_t)(tgt0[t] + g0 + ch) * K + c;
#pragma unroll
    for (int x = 0; x < P; x++) {
      const int q = qmap[(x * P + z) * P + y];
      if (q >= 0) o[3 * q] = add ? o[3 * q] + acc[l][x] : acc[l][x];
    }
  }
}

struct SpecTile {
  int lev, t0, n, pad;   // level entry, first target parent, parents of the tile
};

// Per frequency and tile of target parents: Y[48 x parents] = sum over the
// active directions of A_d X[neighbour].  A wavefront holds the 48 rows of
// 16 parents: row tile i is component i, rows (child a, re/im); lane group
// lk = lane / 16 carries the children 2 lk and 2 lk + 1 of the source parent
// as its k index, 12 contiguous values, so B fragments come straight from
// memory (a neighbour's 384 B row), one direction ahead.  The level's
// operators at this frequency (343 offsets x 6 components, 33 KB) sit in
// LDS; an A fragment is one 16-byte LDS read per (component pair, child
// bit), its real and imaginary part giving the two columns of the pair's
// real form.  An FP64 MFMA occupies the matrix core for 64 cycles, so the
// LDS reads and selects (12 reads per 36 MFMAs) hide behind it.
// Frequencies are dealt to the 8 XCDs, a frequency's tiles following each
// other on one XCD, so its X slab (384 B per source parent) is read from
// that XCD's L2 for the 26 directions.
// WD = 1: the four wavefronts take 16 parents each.  WD = 4: they share 16
// parents and split the directions, partial sums added in wavefront order
// (few parents: four times the workgroups, and no idle wavefronts in the
// tiles of the levels near the root, at a table load per 16 parents).
// Measured WD = 1 / 4 at res 6: 72 parents 0.204 / 0.147 ms, ~460 parents
// 0.525 / 0.552 ms, 4,681 parents 5.9 / 7.3 ms; the whole M2L at 148 and 292
// parents, res 4 102 / 87 and 175 / 153 us, res 8 779 / 651 and 1,245 / 1,329,
// res 10 1,616 / 1,384 and 2,640 / 2,825.  32 parents per wavefront (236
// registers, two wavefronts per SIMD instead of three) was slower
// everywhere: 6.0 ms at 4,681 parents, 0.34 ms at 72.
template <int WD>
__global__ __launch_bounds__(256, 2) void k_spec_gemm(const SpecTile *__restrict__ tiles, int ntiles,
                                                      const double *const *__restrict__ tabs, int f0, int nf,
                                                      const int32_t *__restrict__ nb, int nt, int ns,
                                                      const double *__restrict__ X, double *__restrict__ Y) {
  __shared__ __attribute__((aligned(16))) double tab[343 * 12];
  __shared__ int nbs[4 / WD][26][16];
  const int q = blockIdx.x >> 3;
  const int fr = (int)(blockIdx.x & 7) + 8 * (q / ntiles);
  if (fr >= nf) return;
  const SpecTile tl = tiles[q % ntiles];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int lr = lane & 15, lk = lane >> 4;
  const int col = WD == 1 ? wave : 0, part = WD == 1 ? 0 : wave;  // column group, share of the directions
  {
    const d2v *src = reinterpret_cast<const d2v *>(tabs[tl.lev] + (size_t)(f0 + fr) * (343 * 12));
    d2v *dst = reinterpret_cast<d2v *>(tab);
    for (int i = tid; i < 343 * 6; i += 256) dst[i] = src[i];
  }
  const int w0 = 16 * col;             // first column of this wavefront in the tile
  const int wn = min(16, tl.n - w0);   // its columns (<= 0: none)
  unsigned mask = 0;
  for (int d = 0; d < 26; d++) {
    int v = -1;
    if (lane < wn) v = nb[(size_t)d * nt + tl.t0 + w0 + lane];
    if (__ballot(v >= 0)) mask |= 1u << d;
    if (part == 0 && lane < 16) nbs[col][d][lane] = v < 0 ? ns : v;   // row ns of X is zero
  }
  __syncthreads();
  if (WD == 1 && wn <= 0) return;
  // the next of this wavefront's directions, -1 at the end
  auto next = [&]() {
    int d = -1;
    if (mask) {
      d = __builtin_ctz(mask);
      mask &= mask - 1;
#pragma unroll
      for (int k = 1; k < WD; k++) mask &= mask - 1;
    }
    return d;
  };
  for (int k = 0; k < part; k++) mask &= mask - 1;
  const double *Xf = X + (size_t)fr * (ns + 1) * 48 + lk * 12;
  d4 acc[3];
#pragma unroll
  for (int i = 0; i < 3; i++) acc[i] = d4{0, 0, 0, 0};
  const int a = lr >> 1, rho = lr & 1;
  // offset slot of source child (bx, by, 0) against target child a at direction 0
  const int slot0 = (3 + (lk >> 1) - (a >> 2)) * 49 + (3 + (lk & 1) - ((a >> 1) & 1)) * 7 + 3 - (a & 1);
  const d2v *tabl = reinterpret_cast<const d2v *>(tab) + slot0 * 6;
  d2v bc[6], bn[6];
  auto load = [&](int d, d2v (&v)[6]) {
    const d2v *p = reinterpret_cast<const d2v *>(Xf + (size_t)nbs[col][d][lr] * 48);
#pragma unroll
    for (int s = 0; s < 6; s++) v[s] = p[s];
  };
  auto product = [&](int d, const d2v (&v)[6]) {
    const int e = dir27(d);
    const int ds = 2 * ((e / 9 - 1) * 49 + ((e / 3) % 3 - 1) * 7 + e % 3 - 1);
#pragma unroll
    for (int bl = 0; bl < 2; bl++) {
      const d2v *tp = tabl + (ds + bl) * 6;
      double a0[6], a1[6];
#pragma unroll
      for (int k = 0; k < 6; k++) {
        const d2v t = tp[k];
        a0[k] = rho ? t[1] : t[0];
        a1[k] = rho ? t[0] : -t[1];
      }
      constexpr int sym[3][3] = {{0, 1, 2}, {1, 3, 4}, {2, 4, 5}};
#pragma unroll
      for (int jc = 0; jc < 3; jc++)
#pragma unroll
        for (int i = 0; i < 3; i++)
          acc[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0[sym[i][jc]], v[bl * 3 + jc][0], acc[i], 0, 0, 0);
#pragma unroll
      for (int jc = 0; jc < 3; jc++)
#pragma unroll
        for (int i = 0; i < 3; i++)
          acc[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1[sym[i][jc]], v[bl * 3 + jc][1], acc[i], 0, 0, 0);
    }
  };
  int d = next();
  if (d >= 0) {
    load(d, bc);
    while (true) {
      const int d2 = next();
      if (d2 >= 0) load(d2, bn);
      product(d, bc);
      if (d2 < 0) break;
      d = next();
      if (d >= 0) load(d, bc);
      product(d2, bn);
      if (d < 0) break;
    }
  }
  if constexpr (WD > 1) {  // the operator table is done: its LDS holds the partial sums
    __syncthreads();
    double *ps = tab + (wave - 1) * 768 + lane;
    if (wave > 0) {
#pragma unroll
      for (int i = 0; i < 3; i++)
#pragma unroll
        for (int r = 0; r < 4; r++) ps[(i * 4 + r) * 64] = acc[i][r];
    }
    __syncthreads();
    if (wave > 0) return;
#pragma unroll
    for (int w = 0; w < WD - 1; w++)
#pragma unroll
      for (int i = 0; i < 3; i++)
#pragma unroll
        for (int r = 0; r < 4; r++) acc[i][r] += tab[w * 768 + (i * 4 + r) * 64 + lane];
  }
  if (lr >= wn) return;
  double *Yf = Y + ((size_t)fr * nt + tl.t0 + w0 + lr) * 48;
#pragma unroll
  for (int i = 0; i < 3; i++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int m = lk + 4 * r;
      Yf[(m >> 1) * 6 + i * 2 + (m & 1)] = acc[i][r];
    }
}

std::vector<double> twiddles(int n) {
  std::vector<double> t(2 * n);
  for (int i = 0; i < n; i++) {
    // exact at 0, symmetric about n/2
    const int j = std::min(i, n - i);
    t[2 * i] = std::cos(2.0 * kPi * j / n);
    t[2 * i + 1] = (i == j ? 1.0 : -1.0) * std::sin(2.0 * kPi * j / n);
  }
  return t;
}

template <class F> void with_res(int res, F &&f) {
  switch (res) {
    case 3: f(std::integral_constant<int, 3>()); return;
    case 4: f(std::integral_constant<int, 4>()); return;
    case 5: f(std::integral_constant<int, 5>()); return;
    case 6: f(std::integral_constant<int, 6>()); return;
    case 7: f(std::integral_constant<int, 7>()); return;
    case 8: f(std::integral_constant<int, 8>()); return;
    case 9: f(std::integral_constant<int, 9>()); return;
    case 10: f(std::integral_constant<int, 10>()); return;
  }
  throw Error(NNK_ESTATE, "frequency-space M2L: no transform for this coronaRes");
}

}  // namespace

void spectral_ops(int res, double w, double eps, double mu, SpecOps &out) {
  const int n = 2 * res - 1;
  out.tab.alloc(sizeof(double) * (size_t)spectral_freqs(res) * 343 * 12);
  out.tab.zero();
  DBuf tw;
  tw.upload(twiddles(n));
  with_res(res, [&](auto p) {
    hipLaunchKernelGGL((k_spec_table<decltype(p)::value>), dim3(343, 6), dim3(256), 0, 0, w, eps * eps,
                       1.0 / (8.0 * kPi * mu), tw.as<double>(), out.tab.as<double>());
  });
  NNK_HIP(hipGetLastError());
  NNK_HIP(hipDeviceSynchronize());
}

void plan_spectral_level(const std::vector<int32_t> *cls, const std::vector<int32_t> *gv,
                         const std::vector<int32_t> &parent, const std::vector<int32_t> &child0,
                         const std::vector<uint8_t> &has_src, SpecLevel &L) {
  L.tgt0.clear(); L.tmask.clear(); L.src0.clear(); L.smask.clear(); L.nb.clear();
  L.ok = false;
  L.pairs = L.tile_dirs = 0;
  // target parents in increasing id (Morton) order
  std::vector<int32_t> tpar;
  for (int a = 0; a < 8; a++)
    for (int32_t t : cls[a]) tpar.push_back(parent[t] - 1);
  std::sort(tpar.begin(), tpar.end());
  tpar.erase(std::unique(tpar.begin(), tpar.end()), tpar.end());
  const int nt = (int)tpar.size();
  if (!nt) return;
  L.tgt0.resize(nt);
  L.tmask.assign(nt, 0);
  for (int t = 0; t < nt; t++) L.tgt0[t] = child0[tpar[t]];
  auto tindex = [&](int32_t par) {
    return (int)(std::lower_bound(tpar.begin(), tpar.end(), par) - tpar.begin());
  };
  // neighbours as parent slots first
  std::vector<int32_t> nbp((size_t)26 * nt, -1);
  std::vector<int64_t> want;   // per target parent: pairs counted in the lists
  want.assign(nt, 0);
  for (int a = 0; a < 8; a++) {
    const std::vector<int> sls = class_offset_slots(a);
    const int N = (int)cls[a].size();
    if (!N) continue;
    if (gv[a].size() != sls.size() * (size_t)N) return;
    std::vector<int> ti(N);
    for (int j = 0; j < N; j++) {
      ti[j] = tindex(parent[cls[a][j]] - 1);
      if (L.tgt0[ti[j]] + a != cls[a][j]) return;
      L.tmask[ti[j]] |= 1 << a;
    }
    const int av[3] = {a >> 2, (a >> 1) & 1, a & 1};
    for (size_t b = 0; b < sls.size(); b++) {
      const int o[3] = {sls[b] / 49 - 3, (sls[b] / 7) % 7 - 3, sls[b] % 7 - 3};
      int e = 0, ch = 0;
      for (int k = 0; k < 3; k++) {
        e = 3 * e + ((av[k] + o[k]) >> 1) + 1;
        ch = 2 * ch + ((av[k] + o[k]) & 1);
      }
      const int d = e - (e > 13);
      for (int j = 0; j < N; j++) {
        const int32_t g = gv[a][b * N + j];
        if (g < 0) continue;
        const int32_t par = parent[g] - 1;
        if (e == 13 || child0[par] + ch != g) return;
        int32_t &v = nbp[(size_t)d * nt + ti[j]];
        if (v >= 0 && v != par) return;
        v = par;
        want[ti[j]]++;
      }
    }
  }
  // source parents
  std::vector<int32_t> spar;
  for (int32_t v : nbp)
    if (v >= 0) spar.push_back(v);
  std::sort(spar.begin(), spar.end());
  spar.erase(std::unique(spar.begin(), spar.end()), spar.end());
  const int ns = (int)spar.size();
  L.src0.resize(ns);
  L.smask.assign(ns, 0);
  for (int i = 0; i < ns; i++) {
    L.src0[i] = child0[spar[i]];
    for (int c = 0; c < 8; c++)
      if (has_src[L.src0[i] + c + 1]) L.smask[i] |= 1 << c;
  }
  L.nb.assign((size_t)26 * nt, -1);
  std::vector<int64_t> have(nt, 0);
  for (int d = 0; d < 26; d++) {
    const int e = dir27(d);
    const int dv[3] = {e / 9 - 1, (e / 3) % 3 - 1, e % 3 - 1};
    for (int t = 0; t < nt; t++) {
      const int32_t v = nbp[(size_t)d * nt + t];
      if (v < 0) continue;
      const int i = (int)(std::lower_bound(spar.begin(), spar.end(), v) - spar.begin());
      L.nb[(size_t)d * nt + t] = i;
      for (int a = 0; a < 8; a++) {
        if (!((L.tmask[t] >> a) & 1)) continue;
        for (int c = 0; c < 8; c++) {
          if (!((L.smask[i] >> c) & 1)) continue;
          const int o[3] = {2 * dv[0] + (c >> 2) - (a >> 2), 2 * dv[1] + ((c >> 1) & 1) - ((a >> 1) & 1),
                            2 * dv[2] + (c & 1) - (a & 1)};
          have[t] += std::max({std::abs(o[0]), std::abs(o[1]), std::abs(o[2])}) >= 2;
        }
      }
    }
  }
  // Parents with the same neighbours side by side: a tile of 16 parents
  // walks the directions that any of them has.  (Stable: the interior of a
  // uniform level stays in Morton order.)
  {
    std::vector<uint32_t> m(nt, 0);
    for (int d = 0; d < 26; d++)
      for (int t = 0; t < nt; t++) m[t] |= (uint32_t)(L.nb[(size_t)d * nt + t] >= 0) << d;
    std::vector<int> ord(nt);
    for (int t = 0; t < nt; t++) ord[t] = t;
    std::stable_sort(ord.begin(), ord.end(), [&](int x, int y) { return m[x] > m[y]; });
    auto put = [&](auto &v, size_t off) {
      auto w = std::vector<typename std::decay<decltype(v[0])>::type>(v.begin() + off, v.begin() + off + nt);
      for (int t = 0; t < nt; t++) v[off + t] = w[ord[t]];
    };
    put(L.tgt0, 0);
    put(L.tmask, 0);
    put(have, 0);
    put(want, 0);
    for (int d = 0; d < 26; d++) put(L.nb, (size_t)d * nt);
  }
  // the product sets must be the V lists, pair for pair
  for (int t = 0; t < nt; t++) {
    if (have[t] != want[t]) return;
    L.pairs += have[t];
  }
  for (int d = 0; d < 26; d++)
    for (int t0 = 0; t0 < nt; t0 += 16) {
      bool any = false;
      for (int t = t0; t < std::min(nt, t0 + 16) && !any; t++) any = L.nb[(size_t)d * nt + t] >= 0;
      L.tile_dirs += any;
    }
  L.ok = true;
}

SpectralM2L::SpectralM2L(int res, const std::vector<int32_t> &codes, int K) : res_(res), K_(K) {
  h_qmap_.assign((size_t)res * res * res, -1);
  for (size_t i = 0; i < codes.size(); i++) {
    const int ix = codes[i] & 255, iy = (codes[i] >> 8) & 255, iz = (codes[i] >> 16) & 255;
    h_qmap_[((size_t)ix * res + iz) * res + iy] = (int32_t)i;
  }
}

void SpectralM2L::add(const SpecLevel &L, std::shared_ptr<const SpecOps> ops) {
  if (!L.ok) throw Error(NNK_ESTATE, "frequency-space M2L: unplanned level");
  lev_t0_.push_back(nt_);
  lev_nt_.push_back((int)L.tgt0.size());
  lev_s0_.push_back(ns_);
  h_tgt0_.insert(h_tgt0_.end(), L.tgt0.begin(), L.tgt0.end());
  h_tmask_.insert(h_tmask_.end(), L.tmask.begin(), L.tmask.end());
  h_src0_.insert(h_src0_.end(), L.src0.begin(), L.src0.end());
  h_smask_.insert(h_smask_.end(), L.smask.begin(), L.smask.end());
  h_nb_.push_back(L.nb);
  nt_ += (int)L.tgt0.size();
  ns_ += (int)L.src0.size();
  ops_.push_back(std::move(ops));
}

void SpectralM2L::finish(size_t buf_bytes) {
  if (empty()) return;
  std::vector<int32_t> nb((size_t)26 * nt_, -1);
  std::vector<SpecTile> tiles;
  std::vector<const double *> tab;
  split_ = nt_ < 256;   // see k_spec_gemm: both sides measured
  const int tw = split_ ? 16 : 64;
  for (size_t l = 0; l < ops_.size(); l++) {
    const int t0 = lev_t0_[l], n = lev_nt_[l];
    for (int d = 0; d < 26; d++)
      for (int t = 0; t < n; t++) {
        const int32_t v = h_nb_[l][(size_t)d * n + t];
        nb[(size_t)d * nt_ + t0 + t] = v < 0 ? -1 : v + lev_s0_[l];
      }
    for (int t = 0; t < n; t += tw) tiles.push_back({(int)l, t0 + t, std::min(tw, n - t), 0});
    tab.push_back(ops_[l]->tab.as<double>());
  }
  ntiles_ = (int)tiles.size();
  qmap_.upload(h_qmap_);
  tw_.upload(twiddles(2 * res_ - 1));
  tgt0_.upload(h_tgt0_);
  tmask_.upload(h_tmask_);
  src0_.upload(h_src0_);
  smask_.upload(h_smask_);
  nb_.upload(nb);
  tiles_.upload(tiles);
  tab_.upload(tab);
  const int n = 2 * res_ - 1;
  const size_t per_f = sizeof(double) * 48 * ((size_t)ns_ + 1 + nt_);
  kx_step_ = res_;
  while (kx_step_ > 1 && per_f * (size_t)n * n * kx_step_ > buf_bytes) kx_step_--;
  const size_t nf = std::min<size_t>(spectral_freqs(res_), (size_t)n * n * kx_step_);
  X_.alloc(sizeof(double) * 48 * nf * ((size_t)ns_ + 1));
  Y_.alloc(sizeof(double) * 48 * nf * (size_t)nt_);
  X_.zero();   // row ns_ of every frequency stays zero (absent neighbours)
  h_nb_.clear();
}

void SpectralM2L::run(const double *up, double *chk, hipStream_t s) const {
  with_res(res_, [&](auto p) {
    constexpr int P = decltype(p)::value, n = 2 * P - 1;
    constexpr int T = P <= 8 ? 256 : 512;
    for (int kx0 = 0; kx0 < P; kx0 += kx_step_) {
      const int nkx = std::min(kx_step_, P - kx0);
      const int f0 = plane_base(P, kx0), f1 = kx0 + nkx == P ? (n * n * n + 1) / 2 : plane_base(P, kx0 + nkx);
      const int nf = f1 - f0;
      if (ns_) {
        // few parents: the planes side by side, a workgroup each; many: all planes by
        // one workgroup, which reads the densities once.  The whole M2L in us, side by
        // side / all by one: 72 parents res 6 172 / 182, res 10 832 / 828; 292 res 6 508 /
        // 511, res 10 2,635 / 2,496; 916 1,280 / 1,247 and 7,122 / 6,586; 1,172 1,625 /
        // 1,596 and 9,055 / 7,991; 4,681 res 6 6,747 / 6,310.  (The sides meet near 300
        // parents at res 6; up to the line at 1,024 that is 2 to 8 % of the M2L.)
        const int kxn = ns_ < 1024 ? 1 : nkx;
        hipLaunchKernelGGL((k_spec_fwd<P, T>), dim3(ns_, (nkx + kxn - 1) / kxn), dim3(T), 0, s, up, K_,
                           src0_.as<int32_t>(), smask_.as<int32_t>(), qmap_.as<int32_t>(), tw_.as<double>(), kx0, nkx,
                           kxn, X_.as<double>(), (size_t)48 * (ns_ + 1));
        NNK_HIP(hipGetLastError());
      }
      const dim3 grid((unsigned)(8 * ((nf + 7) / 8) * ntiles_));
      auto gemm = [&](auto kern) {
        hipLaunchKernelGGL(kern, grid, dim3(256), 0, s, tiles_.as<SpecTile>(), ntiles_, tab_.as<const double *>(), f0,
                           nf, nb_.as<int32_t>(), nt_, ns_, X_.as<double>(), Y_.as<double>());
      };
      if (split_) gemm(k_spec_gemm<4>);
      else gemm(k_spec_gemm<1>);
      NNK_HIP(hipGetLastError());
      auto inv = [&](auto cg) {
        constexpr int CG = decltype(cg)::value;
        hipLaunchKernelGGL((k_spec_inv<P, CG, T>), dim3((unsigned)(nt_ * (8 / CG))), dim3(T), 0, s, Y_.as<double>(),
                           (size_t)48 * nt_, K_, tgt0_.as<int32_t>(), tmask_.as<int32_t>(), qmap_.as<int32_t>(),
                           tw_.as<double>(), kx0, nkx, kx0 > 0 ? 1 : 0, chk);
      };
      // 2 children a workgroup / 8, the whole M2L in us: 72 parents res 6 171 / 181, res
      // 10 832 / 808; 292 509 / 506 and 2,644 / 2,554; 916 1,283 / 1,261 and 7,128 /
      // 6,728; 1,172 1,608 / 1,595 and 8,483 / 7,985; 4,681 res 6 6,455 / 6,310
      if (nt_ < 1024) inv(std::integral_constant<int, 2>());
      else inv(std::integral_constant<int, 8>());
      NNK_HIP(hipGetLastError());
    }
  });
}

}  // namespace nnk
