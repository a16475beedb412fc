// Device kernels for the KIFMM matvec (FP64 form).
//
// Notation: a node's "up surface" is the res^3 grid on its box minus the
// interior, its "down surface" the same on the box widened by its width on
// every side (Tools/KIFMM/genupsurf.m, gendownsurf.m).  Surface point p has
// grid indices packed in surf_idx[p] = ix | iy<<8 | iz<<16, ordered y
// fastest, then x, then z.  Densities are stored per node as 3*Nq doubles,
// interleaved [p0x p0y p0z p1x ...] as in the reference's uppot(node,:).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace nnk {

constexpr double kPi = 3.14159265358979323846;

// linspace(d1,d2,n)(k): d1 + (k*(d2-d1))/(n-1) with exact endpoints, as
// MATLAB's linspace computes it.
__device__ __forceinline__ double lin(double d1, double d2, int k, int n1) {
  if (k == 0) return d1;
  if (k == n1) return d2;
  return d1 + ((double)k * (d2 - d1)) / (double)n1;
}

__device__ __forceinline__ void surf_point(const double *__restrict__ box, int down, int code,
                                           int n1, double &x, double &y, double &z) {
  double lo0 = box[0], lo1 = box[1], lo2 = box[2], hi0 = box[3], hi1 = box[4], hi2 = box[5];
  if (down) {
    double w0 = hi0 - lo0, w1 = hi1 - lo1, w2 = hi2 - lo2;
    lo0 = lo0 - w0; hi0 = hi0 + w0;
    lo1 = lo1 - w1; hi1 = hi1 + w1;
    lo2 = lo2 - w2; hi2 = hi2 + w2;
  }
  x = lin(lo0, hi0, code & 255, n1);
  y = lin(lo1, hi1, (code >> 8) & 255, n1);
  z = lin(lo2, hi2, (code >> 16) & 255, n1);
}

// u += S(t <- s) q without the 1/(8 pi mu) factor:
// S q = [(r^2 + 2 eps^2) q + r (r.q)] / (r^2 + eps^2)^{3/2},  r = t - s.
__device__ __forceinline__ void stokeslet_acc(double tx, double ty, double tz, double sx, double sy,
                                              double sz, double qx, double qy, double qz, double e2,
                                              double &ux, double &uy, double &uz) {
  double rx = tx - sx, ry = ty - sy, rz = tz - sz;
  double r2 = rx * rx + ry * ry + rz * rz;
  double re = r2 + e2;
  double inv = rsqrt(re);
  double inv3 = inv * inv * inv;
  double iso = (re + e2) * inv3;
  double rq = (rx * qx + ry * qy + rz * qz) * inv3;
  ux += iso * qx + rq * rx;
  uy += iso * qy + rq * ry;
  uz += iso * qz + rq * rz;
}

// 1 / sqrt(x) for x > 0: the hardware estimate (relative error below 2^-22)
// and one third-order step, y (1 + e/2 + 3 e^2 / 8) with e = 1 - x y^2, whose
// own error is of order e^3.  (x = 0 and x = inf give NaN: the kernel's sums
// are NaN there with any reciprocal square root.)
__device__ __forceinline__ double rsqrt_pos(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = __builtin_fma(-(x * y), y, 1.0);
  return __builtin_fma(y * e, __builtin_fma(e, 0.375, 0.5), y);
}

// stokeslet_acc in 28 FP64 instruction slots (the hardware estimate counts
// four): r^2 + eps^2 as one chain, the isotropic factor
// (r^2 + 2 eps^2) / (r^2 + eps^2)^{3/2} as 1/s + eps^2 / s^3.  For the FP64
// kernels whose sources or targets are wavefront-uniform (scalar operands),
// so that nothing but these slots is issued per pair.
__device__ __forceinline__ void stokeslet_acc64(double tx, double ty, double tz, double sx, double sy, double sz,
                                                double qx, double qy, double qz, double e2, double &ux, double &uy,
                                                double &uz) {
  const double rx = tx - sx, ry = ty - sy, rz = tz - sz;
  const double re = __builtin_fma(rx, rx, __builtin_fma(ry, ry, __builtin_fma(rz, rz, e2)));
  const double inv = rsqrt_pos(re);
  const double inv3 = inv * inv * inv;
  const double iso = __builtin_fma(e2, inv3, inv);
  const double rq = __builtin_fma(rx, qx, __builtin_fma(ry, qy, rz * qz)) * inv3;
  ux = __builtin_fma(iso, qx, __builtin_fma(rq, rx, ux));
  uy = __builtin_fma(iso, qy, __builtin_fma(rq, ry, uy));
  uz = __builtin_fma(iso, qz, __builtin_fma(rq, rz, uz));
}

// The terms of stokeslet_acc of the N sources v[6 k ..] (position, strength),
// stage by stage so that their dependent chains overlap, every rounding
// written out: the sums of batched solves keep the roundings they were
// defined with (their GMRES turns a last-bit change into 1e-8 of the
// solution), whatever the compiler contracts elsewhere.
template <int N>
__device__ __forceinline__ void stokeslet_terms_fixed(double tx, double ty, double tz, const double (&v)[6 * N],
                                                      double e2, double (&rx)[N], double (&ry)[N], double (&rz)[N]) {
#pragma clang fp contract(off)
  double re[N], y[N], e[N], rq[N], iso[N];
#pragma unroll
  for (int k = 0; k < N; k++) {
    rx[k] = tx - v[6 * k];
    ry[k] = ty - v[6 * k + 1];
    rz[k] = tz - v[6 * k + 2];
  }
#pragma unroll
  for (int k = 0; k < N; k++) re[k] = ry[k] * ry[k];
#pragma unroll
  for (int k = 0; k < N; k++) re[k] = __builtin_fma(rx[k], rx[k], re[k]);
#pragma unroll
  for (int k = 0; k < N; k++) re[k] = __builtin_fma(rz[k], rz[k], re[k]);
#pragma unroll
  for (int k = 0; k < N; k++) re[k] = re[k] + e2;
#pragma unroll
  for (int k = 0; k < N; k++) y[k] = __builtin_amdgcn_rsq(re[k]);
#pragma unroll
  for (int k = 0; k < N; k++) rq[k] = ry[k] * v[6 * k + 4];
#pragma unroll
  for (int k = 0; k < N; k++) rq[k] = __builtin_fma(rx[k], v[6 * k + 3], rq[k]);
#pragma unroll
  for (int k = 0; k < N; k++) rq[k] = __builtin_fma(rz[k], v[6 * k + 5], rq[k]);
#pragma unroll
  for (int k = 0; k < N; k++) e[k] = re[k] * y[k];
#pragma unroll
  for (int k = 0; k < N; k++) e[k] = __builtin_fma(-e[k], y[k], 1.0);
#pragma unroll
  for (int k = 0; k < N; k++) iso[k] = re[k] + e2;
#pragma unroll
  for (int k = 0; k < N; k++) re[k] = __builtin_fma(e[k], 0.375, 0.5);
#pragma unroll
  for (int k = 0; k < N; k++) e[k] = y[k] * e[k];
#pragma unroll
  for (int k = 0; k < N; k++) y[k] = __builtin_fma(e[k], re[k], y[k]);
#pragma unroll
  for (int k = 0; k < N; k++) re[k] = y[k] * y[k];
#pragma unroll
  for (int k = 0; k < N; k++) y[k] = y[k] * re[k];
#pragma unroll
  for (int k = 0; k < N; k++) {
    iso[k] = iso[k] * y[k];
    rq[k] = rq[k] * y[k];
  }
#pragma unroll
  for (int k = 0; k < N; k++) {
    rx[k] = __builtin_fma(v[6 * k + 3], iso[k], rx[k] * rq[k]);
    ry[k] = __builtin_fma(v[6 * k + 4], iso[k], ry[k] * rq[k]);
    rz[k] = __builtin_fma(v[6 * k + 5], iso[k], rz[k] * rq[k]);
  }
}

// Mixed form: the separation r = t - s is formed in FP64 (so near pairs keep
// their digits), the kernel is evaluated in FP32 with the hardware reciprocal
// square root, and the result is accumulated in FP64.  The strength comes in
// FP32 (rounded once, where the source is staged).
__device__ __forceinline__ void stokeslet_acc_f32q(double tx, double ty, double tz, double sx,
                                                   double sy, double sz, float fx, float fy,
                                                   float fz, double e2, double &ux, double &uy,
                                                   double &uz) {
  const float rx = (float)(tx - sx), ry = (float)(ty - sy), rz = (float)(tz - sz);
  const float e2f = (float)e2;
  const float r2 = rx * rx + ry * ry + rz * rz;
  const float re = r2 + e2f;
  const float inv = __builtin_amdgcn_rsqf(re);
  const float inv3 = inv * inv * inv;
  const float iso = __builtin_fmaf(e2f, inv3, inv);  // (re + e2) / re^1.5
  const float rq = (rx * fx + ry * fy + rz * fz) * inv3;
  ux += (double)(iso * fx + rq * rx);
  uy += (double)(iso * fy + rq * ry);
  uz += (double)(iso * fz + rq * rz);
}

// the FP32 term of one source (stokeslet_acc_f32q before its FP64 addition),
// every rounding written out
__device__ __forceinline__ void stokeslet_term_f32_fixed(double tx, double ty, double tz, double sx, double sy,
                                                         double sz, float fx, float fy, float fz, float e2f, float &gx,
                                                         float &gy, float &gz) {
#pragma clang fp contract(off)
  const float rx = (float)(tx - sx), ry = (float)(ty - sy), rz = (float)(tz - sz);
  const float re = __builtin_fmaf(rz, rz, __builtin_fmaf(rx, rx, ry * ry)) + e2f;
  const float inv = __builtin_amdgcn_rsqf(re);
  const float inv3 = inv * (inv * inv);
  const float iso = __builtin_fmaf(e2f, inv3, inv);  // (re + e2) / re^1.5
  const float rq = __builtin_fmaf(rz, fz, __builtin_fmaf(rx, fx, ry * fy)) * inv3;
  gx = __builtin_fmaf(fx, iso, rq * rx);
  gy = __builtin_fmaf(fy, iso, rq * ry);
  gz = __builtin_fmaf(fz, iso, rq * rz);
}

// FP32-math forms: LDS stage of up to T sources, positions in FP64, strengths
// rounded to FP32 once when staged (the values the pair routine would
// otherwise round per pair).  acc(j, ...) adds source j.
template <int T> struct SrcStage {
  double p[3 * T];
  __attribute__((aligned(16))) float q[4 * T];
  __device__ __forceinline__ void put(int i, double x, double y, double z, double qx, double qy, double qz) {
    p[3 * i] = x; p[3 * i + 1] = y; p[3 * i + 2] = z;
    q[4 * i] = (float)qx; q[4 * i + 1] = (float)qy; q[4 * i + 2] = (float)qz;
  }
  __device__ __forceinline__ void acc(int j, double tx, double ty, double tz, double e2, double &ux,
                                      double &uy, double &uz) const {
    stokeslet_acc_f32q(tx, ty, tz, p[3 * j], p[3 * j + 1], p[3 * j + 2], q[4 * j], q[4 * j + 1], q[4 * j + 2],
                       e2, ux, uy, uz);
  }
  // sources j = j0, j0 + step, ... < cnt, four per iteration: the four
  // FP32 contributions are added in FP32 (in order) and then once into the
  // FP64 sums, which saves three conversions and FP64 adds per pair
  __device__ __forceinline__ void run(int j0, int step, int cnt, double tx, double ty, double tz, double e2,
                                      double &ux, double &uy, double &uz) const {
    const float e2f = (float)e2;
    int j = j0;
    for (; j + 3 * step < cnt; j += 4 * step) {
      float gx = 0.f, gy = 0.f, gz = 0.f;
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const int i = j + k * step;
        const float4 f = *reinterpret_cast<const float4 *>(&q[4 * i]);
        const float rx = (float)(tx - p[3 * i]), ry = (float)(ty - p[3 * i + 1]), rz = (float)(tz - p[3 * i + 2]);
        const float r2 = rx * rx + ry * ry + rz * rz;
        const float re = r2 + e2f;
        const float inv = __builtin_amdgcn_rsqf(re);
        const float inv3 = inv * inv * inv;
        const float iso = __builtin_fmaf(e2f, inv3, inv);  // (re + e2) / re^1.5
        const float rq = (rx * f.x + ry * f.y + rz * f.z) * inv3;
        gx += iso * f.x + rq * rx;
        gy += iso * f.y + rq * ry;
        gz += iso * f.z + rq * rz;
      }
      ux += (double)gx;
      uy += (double)gy;
      uz += (double)gz;
    }
    for (; j < cnt; j += step) acc(j, tx, ty, tz, e2, ux, uy, uz);
  }
};

// FP32-math stage for the evaluations that involve a surface (S2M, P2L,
// L2T, M2T): positions are FP32 offsets from an origin o, formed in FP64
// and rounded once (at staging for the sources, per target for the
// targets).  The separation t - s is then one FP32 subtraction.  Its
// rounding error is at most 2^-24 (|t - o| + |s - o|) per component.
// The callers put o at the centre of the smaller of the two boxes (width
// w).  The surface geometry keeps every such pair at least w apart and the
// point nearer o within 1.5 sqrt(3) w of it, so the error stays within a
// few FP32 ulps of |r|, the size of the kernel's own FP32 rounding.  (P2P
// pairs can be arbitrarily close and keep the FP64 separation of
// SrcStage.)
template <int T> struct SrcStageRel {
  float4 p[T];  // x, y, z offset from the origin; w unused
  float4 q[T];  // strength; w unused
  __device__ __forceinline__ void put(int i, double dx, double dy, double dz, double qx, double qy,
                                      double qz) {
    p[i] = float4{(float)dx, (float)dy, (float)dz, 0.f};
    q[i] = float4{(float)qx, (float)qy, (float)qz, 0.f};
  }
  __device__ __forceinline__ static void pair(const float4 &s, const float4 &f, float tx, float ty, float tz,
                                              float e2f, float &gx, float &gy, float &gz) {
    const float rx = tx - s.x, ry = ty - s.y, rz = tz - s.z;
    const float r2 = rx * rx + ry * ry + rz * rz;
    const float re = r2 + e2f;
    const float inv = __builtin_amdgcn_rsqf(re);
    const float inv3 = inv * inv * inv;
    const float iso = __builtin_fmaf(e2f, inv3, inv);  // (re + e2) / re^1.5
    const float rq = (rx * f.x + ry * f.y + rz * f.z) * inv3;
    gx = __builtin_fmaf(rq, rx, __builtin_fmaf(iso, f.x, gx));
    gy = __builtin_fmaf(rq, ry, __builtin_fmaf(iso, f.y, gy));
    gz = __builtin_fmaf(rq, rz, __builtin_fmaf(iso, f.z, gz));
  }
  // sources j = j0, j0 + step, ... < cnt onto the target offset (tx, ty,
  // tz): each group of four is summed in FP32, then added to the FP64 sums
  __device__ __forceinline__ void run(int j0, int step, int cnt, float tx, float ty, float tz, float e2f,
                                      double &ux, double &uy, double &uz) const {
    int j = j0;
    for (; j + 3 * step < cnt; j += 4 * step) {
      float gx = 0.f, gy = 0.f, gz = 0.f;
#pragma unroll
      for (int k = 0; k < 4; k++) pair(p[j + k * step], q[j + k * step], tx, ty, tz, e2f, gx, gy, gz);
      ux += (double)gx;
      uy += (double)gy;
      uz += (double)gz;
    }
    for (; j < cnt; j += step) {
      float gx = 0.f, gy = 0.f, gz = 0.f;
      pair(p[j], q[j], tx, ty, tz, e2f, gx, gy, gz);
      ux += (double)gx;
      uy += (double)gy;
      uz += (double)gz;
    }
  }
};

// centre of box [lo0 lo1 lo2 hi0 hi1 hi2]
__device__ __forceinline__ void box_centre(const double *__restrict__ box, double &cx, double &cy, double &cz) {
  cx = 0.5 * (box[0] + box[3]);
  cy = 0.5 * (box[1] + box[4]);
  cz = 0.5 * (box[2] + box[5]);
}

}  // namespace nnk
