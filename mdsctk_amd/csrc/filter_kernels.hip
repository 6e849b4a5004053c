// gfx950 kernels of the tile filter: which (reference pair, fit block) tiles
// of a fitted query can hold a candidate at all.
//
// A query's contraction spends 27 MFMAs (split forms) per 16 atoms on every
// 32 x 32 tile of frame pairs, but with thresholds already set (a landmark
// pass, a band pass) nearly every tile of a set in landmark order holds only
// pairs far past both frames' thresholds.  The filter proves that from one
// BF16 product (9 MFMAs), and often from the first quarter of the atoms, and
// the contraction then runs over the tiles that are left.
//
// The bound.  Every frame is turned onto one mean structure m by optimal
// superposition: x_a = sqrt(w) R_a (x - c) = m + d_a.  Then
//   M = sum_i x_a x_b^T = C + P_a + P_b^T + sum_i d_a d_b^T,
//   C = sum m m^T,  P_a = sum d_a m^T,
// and only the last term is rounded: h = bf16(d), l = d - h,
//   M1 = C + P_a + P_b^T + sum h_a h_b^T,
//   |lambda(M) - lambda(M1)| <= |d_a| |l_b| + |l_a| max(|d_b|, |h_b|),
// because lambda(M) = max over rotations R of tr(R M) and |tr(R sum u v^T)|
// <= |u| |v|.  The norms are those of the frame's actual remainders, so the
// bound is proven, not fitted; d is small against x for frames of one
// system, which is what makes one BF16 product enough.  With
// lambda(M1) <= the sum of M1's column norms, a pair is past both
// thresholds when
//   sum of column norms + errors < (G_a + G_b - T) / 2.
// The P terms ride along as 12 extra "atoms" (P as two BF16 halves against
// unit vectors, on either side), C is the accumulators' start value.
//
// A first segment of the atoms (about a quarter, spread over the frame)
// bounds the rest by Cauchy-Schwarz: lambda(M) <= lambda(M') + |x''_a||x''_b|.
//
// Measured, self query of 200000 x 1000 atoms, k = 64 (50 metastable
// states): the contraction over every tile took 917 ms; the filter took
// 91 ms over all tiles (1 PFLOP/s of BF16, what a large matrix product reaches
// on this card is 1.1), takes 31 ms over those that the ball test (kOutBall)
// leaves, and leaves 2.3 % of the tiles, which take 31 ms.  Without the first
// segment the filter alone took over 220 ms.  Cross query of 4096
// against 100000 x 500 atoms, k = 50 (one basin): contraction 10.0 ms before;
// the filter takes 4.0 ms (1.1 PFLOP/s) and leaves tiles for 2.1 ms.  50000
// against 50000 x 304 atoms in plain FP32, k = 100: 124 ms before, now 6 for
// the landmarks and places, 14 for the filter and 25 for the tiles left.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <climits>
#include <cmath>

#include "frame_math.h"
#include "knn_device.h"

namespace mdsctk {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) void lds_void_t;

// Rotation R (row-major) maximising tr(R^T S') for S = sum w x m^T, i.e. R x
// closest to m: the eigenvector of the largest eigenvalue of Horn's 4x4 key
// matrix by cyclic Jacobi in FP64, as a unit quaternion.  It need not be
// exact: any proper rotation leaves every score unchanged.
__device__ void superpose(const double* S, double* R) {
  const double xx = S[0], xy = S[1], xz = S[2], yx = S[3], yy = S[4], yz = S[5];
  const double zx = S[6], zy = S[7], zz = S[8];
  double a[4][4], v[4][4];
  a[0][0] = xx + yy + zz; a[1][1] = xx - yy - zz; a[2][2] = -xx + yy - zz; a[3][3] = -xx - yy + zz;
  a[0][1] = a[1][0] = yz - zy;
  a[0][2] = a[2][0] = zx - xz;
  a[0][3] = a[3][0] = xy - yx;
  a[1][2] = a[2][1] = xy + yx;
  a[1][3] = a[3][1] = zx + xz;
  a[2][3] = a[3][2] = yz + zy;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) v[i][j] = i == j;
  const double scale = fabs(xx) + fabs(xy) + fabs(xz) + fabs(yx) + fabs(yy) + fabs(yz) + fabs(zx) +
                       fabs(zy) + fabs(zz);
  for (int sweep = 0; sweep < 10; ++sweep) {
    double off = 0.0;
#pragma unroll
    for (int p = 0; p < 3; ++p)
#pragma unroll
      for (int q = p + 1; q < 4; ++q) off += fabs(a[p][q]);
    if (!(off > 1e-9 * scale)) break;
#pragma unroll
    for (int p = 0; p < 3; ++p)
#pragma unroll
      for (int q = p + 1; q < 4; ++q) {
        const double apq = a[p][q];
        if (fabs(apq) <= 1e-18 * scale) continue;
        const double th = (a[q][q] - a[p][p]) / (2.0 * apq);
        double t = 1.0 / (fabs(th) + sqrt(th * th + 1.0));
        if (th < 0.0) t = -t;
        const double c = 1.0 / sqrt(t * t + 1.0), s = t * c;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const double akp = a[k][p], akq = a[k][q];
          a[k][p] = c * akp - s * akq;
          a[k][q] = s * akp + c * akq;
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const double apk = a[p][k], aqk = a[q][k];
          a[p][k] = c * apk - s * aqk;
          a[q][k] = s * apk + c * aqk;
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const double vkp = v[k][p], vkq = v[k][q];
          v[k][p] = c * vkp - s * vkq;
          v[k][q] = s * vkp + c * vkq;
        }
      }
  }
  double best = a[0][0], q0 = v[0][0], q1 = v[1][0], q2 = v[2][0], q3 = v[3][0];
#pragma unroll
  for (int j = 1; j < 4; ++j)
    if (a[j][j] > best) {
      best = a[j][j];
      q0 = v[0][j]; q1 = v[1][j]; q2 = v[2][j]; q3 = v[3][j];
    }
  const double nq = q0 * q0 + q1 * q1 + q2 * q2 + q3 * q3;
  if (!(nq > 0.5 && nq < 2.0)) { q0 = 1.0; q1 = q2 = q3 = 0.0; }  // non-finite input
  const double in = (nq > 0.5 && nq < 2.0) ? 1.0 / nq : 1.0;
  R[0] = (q0 * q0 + q1 * q1 - q2 * q2 - q3 * q3) * in;
  R[1] = 2 * (q1 * q2 - q0 * q3) * in;
  R[2] = 2 * (q1 * q3 + q0 * q2) * in;
  R[3] = 2 * (q1 * q2 + q0 * q3) * in;
  R[4] = (q0 * q0 - q1 * q1 + q2 * q2 - q3 * q3) * in;
  R[5] = 2 * (q2 * q3 - q0 * q1) * in;
  R[6] = 2 * (q1 * q3 - q0 * q2) * in;
  R[7] = 2 * (q2 * q3 + q0 * q1) * in;
  R[8] = (q0 * q0 - q1 * q1 - q2 * q2 + q3 * q3) * in;
}

__device__ __forceinline__ void rotate3(const double* R, double e0, double e1, double e2, double* o) {
  o[0] = fma(R[2], e2, fma(R[1], e1, R[0] * e0));
  o[1] = fma(R[5], e2, fma(R[4], e1, R[3] * e0));
  o[2] = fma(R[8], e2, fma(R[7], e1, R[6] * e0));
}

// ---------------------------------------------------------------------------
// the mean structure: kFilterSamples frames spread over the set, turned onto
// frame 0 and averaged, in the average's own axes and scaled by sqrt(w).

// One wave per sample: its centroid and rotation onto frame 0 (12 doubles).
__global__ __launch_bounds__(256) void mean_align_kernel(const float* __restrict__ xyz, int64_t n,
                                                         int natoms, const float* __restrict__ w,
                                                         double W, int samples,
                                                         double* __restrict__ al) {
  const int s = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (s >= samples) return;
  const F3* x = reinterpret_cast<const F3*>(xyz) + (int64_t)s * n / samples * natoms;
  const F3* b = reinterpret_cast<const F3*>(xyz);
  double c[3] = {0, 0, 0}, cb[3] = {0, 0, 0}, S[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  for (int i = lane; i < natoms; i += 64) {
    const double wi = w[i];
    const double a[3] = {x[i].x, x[i].y, x[i].z}, q[3] = {b[i].x, b[i].y, b[i].z};
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      c[k] += wi * a[k];
      cb[k] += wi * q[k];
#pragma unroll
      for (int l = 0; l < 3; ++l) S[3 * k + l] += wi * a[k] * q[l];
    }
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    c[k] = wave_sum_d(c[k]) / W;
    cb[k] = wave_sum_d(cb[k]) / W;
  }
#pragma unroll
  for (int k = 0; k < 9; ++k) S[k] = wave_sum_d(S[k]) - W * c[k / 3] * cb[k % 3];
  double R[9];
  superpose(S, R);
  if (lane < 12) al[s * 12 + lane] = lane < 9 ? R[lane] : c[lane - 9];
}

// One thread per atom: the average over the samples.
__global__ __launch_bounds__(64) void mean_sum_kernel(const float* __restrict__ xyz, int64_t n,
                                                      int natoms, int samples,
                                                      const double* __restrict__ al,
                                                      double* __restrict__ mean) {
  const int i = blockIdx.x * 64 + threadIdx.x;
  if (i >= natoms) return;
  double m[3] = {0, 0, 0};
#pragma unroll 8
  for (int s = 0; s < samples; ++s) {
    const F3 v = (reinterpret_cast<const F3*>(xyz) + (int64_t)s * n / samples * natoms)[i];
    const double* A = al + s * 12;
    double o[3];
    rotate3(A, (double)v.x - A[9], (double)v.y - A[10], (double)v.z - A[11], o);
    m[0] += o[0];
    m[1] += o[1];
    m[2] += o[2];
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) mean[3 * i + k] = m[k] / samples;
}

// The atom's slot in the filter operand: the first segment takes n0 atoms
// spread evenly over the frame, the second the others in order.
__device__ __forceinline__ int atoms_before(int a, int n0, int natoms) {
  return (int)(((int64_t)a * n0 + natoms - 1) / natoms);  // members of segment 0 below a
}
__device__ __forceinline__ bool in_first(int a, int n0, int natoms) {
  return atoms_before(a + 1, n0, natoms) > atoms_before(a, n0, natoms);
}

// Axes of a symmetric 3x3 (xx, xy, xz, yy, yz, zz) as the rows of a proper
// rotation, by decreasing eigenvalue (cyclic Jacobi).
__device__ void axes3(const double* t, double* Q) {
  double a[3][3] = {{t[0], t[1], t[2]}, {t[1], t[3], t[4]}, {t[2], t[4], t[5]}};
  double v[3][3] = {{1, 0, 0}, {0, 1, 0}, {0, 0, 1}};
  for (int sweep = 0; sweep < 12; ++sweep) {
    const double off = fabs(a[0][1]) + fabs(a[0][2]) + fabs(a[1][2]);
    if (!(off > 1e-15 * (fabs(a[0][0]) + fabs(a[1][1]) + fabs(a[2][2])))) break;
    for (int pq = 0; pq < 3; ++pq) {
      const int p = pq == 2 ? 1 : 0, r = pq == 0 ? 1 : 2;
      if (a[p][r] == 0.0) continue;
      const double th = (a[r][r] - a[p][p]) / (2.0 * a[p][r]);
      double u = 1.0 / (fabs(th) + sqrt(th * th + 1.0));
      if (th < 0.0) u = -u;
      const double cs = 1.0 / sqrt(u * u + 1.0), sn = u * cs;
      for (int k = 0; k < 3; ++k) {
        const double x = a[k][p], y = a[k][r];
        a[k][p] = cs * x - sn * y;
        a[k][r] = sn * x + cs * y;
      }
      for (int k = 0; k < 3; ++k) {
        const double x = a[p][k], y = a[r][k], vx = v[k][p], vy = v[k][r];
        a[p][k] = cs * x - sn * y;
        a[r][k] = sn * x + cs * y;
        v[k][p] = cs * vx - sn * vy;
        v[k][r] = sn * vx + cs * vy;
      }
    }
  }
  int o[3] = {0, 1, 2};
  for (int i = 0; i < 2; ++i)
    for (int j = 0; j < 2 - i; ++j)
      if (a[o[j]][o[j]] < a[o[j + 1]][o[j + 1]]) {
        const int x = o[j];
        o[j] = o[j + 1];
        o[j + 1] = x;
      }
  for (int i = 0; i < 3; ++i) {
    Q[i] = v[i][o[0]];
    Q[3 + i] = v[i][o[1]];
  }
  Q[6] = Q[1] * Q[5] - Q[2] * Q[4];
  Q[7] = Q[2] * Q[3] - Q[0] * Q[5];
  Q[8] = Q[0] * Q[4] - Q[1] * Q[3];
}

__device__ double block_sum(double v, double* red) {
  v = wave_sum_d(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double s = 0.0;
  for (int k = 0; k < (int)(blockDim.x >> 6); ++k) s += red[k];
  return s;
}

// One workgroup: the mean in its axes, scaled by sqrt(w), its segments' C
// (FP32, row-major) and norms, and the slot map (atom, -1 padding, -2-j the
// j-th extra slot of a segment).
__global__ __launch_bounds__(256) void mean_final_kernel(const float* __restrict__ w,
                                                         const float* __restrict__ sw, int natoms,
                                                         FilterShape sh, double* __restrict__ mean,
                                                         FilterMean* __restrict__ mc,
                                                         int* __restrict__ slots) {
  __shared__ double red[4];
  const int tid = threadIdx.x;
  double t[6] = {0, 0, 0, 0, 0, 0};
  for (int i = tid; i < natoms; i += 256) {
    const double wi = w[i], x = mean[3 * i], y = mean[3 * i + 1], z = mean[3 * i + 2];
    t[0] += wi * x * x; t[1] += wi * x * y; t[2] += wi * x * z;
    t[3] += wi * y * y; t[4] += wi * y * z; t[5] += wi * z * z;
  }
  for (int k = 0; k < 6; ++k) t[k] = block_sum(t[k], red);
  double Q[9];
  axes3(t, Q);
  double C[2][9] = {};
  for (int i = tid; i < natoms; i += 256) {
    double m[3];
    rotate3(Q, mean[3 * i], mean[3 * i + 1], mean[3 * i + 2], m);
    const int seg = (sh.u1 && !in_first(i, sh.n0, natoms)) ? 1 : 0;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      m[k] *= (double)sw[i];
      mean[3 * i + k] = m[k];
    }
#pragma unroll
    for (int k = 0; k < 9; ++k) {
      C[0][k] += seg ? 0.0 : m[k / 3] * m[k % 3];
      C[1][k] += seg ? m[k / 3] * m[k % 3] : 0.0;
    }
  }
  for (int s = 0; s < 2; ++s)
    for (int k = 0; k < 9; ++k) {
      const double v = block_sum(C[s][k], red);
      if (tid == 0) mc->C[s][k] = (float)v;
      C[s][k] = v;
    }
  if (tid == 0) {
    const double q0 = C[0][0] + C[0][4] + C[0][8], q1 = C[1][0] + C[1][4] + C[1][8];
    mc->norm0 = sqrt(q0);
    mc->norm = sqrt(q0 + q1);
  }
  const int g0 = sh.segment_slots(0), total = sh.slots();
  for (int s = tid; s < total; s += 256) {
    const int seg = s >= g0, len = sh.segment_slots(seg), at = s - (seg ? g0 : 0);
    slots[s] = at >= len - kFilterExtra ? -2 - (at - (len - kFilterExtra)) : -1;
  }
  __syncthreads();
  for (int a = tid; a < natoms; a += 256) {
    const int before = sh.u1 ? atoms_before(a, sh.n0, natoms) : a;
    const bool first = !sh.u1 || in_first(a, sh.n0, natoms);
    slots[first ? before : g0 + a - before] = a;
  }
}

// ---------------------------------------------------------------------------
// per-frame terms and operand

// One wave per row (row f holds frame perm[f], or f): centroid, rotation
// onto the mean, and the row's terms of the bound.
//   full: x = G/2 less the row's own errors, y = max(|d|, |h|), z = |l|, w = 0
//   pre:  the same over the first segment; w = |x''| over the second
// The FP32 accumulation of a chain of s MFMAs is allowed 2^-22 of the
// largest partial sum per step in every entry (5.2 bounds the nuclear norm
// of a 3x3 matrix of such entries); every partial sum is at most
// (|m| + |d_a|)(|m| + |d_b|) <= the mean of the squares.
__global__ __launch_bounds__(256) void filter_stats_kernel(
    const float* __restrict__ xyz, int64_t n, int64_t rows, int natoms,
    const float* __restrict__ w, const float* __restrict__ sw, double W,
    const double* __restrict__ mean, const FilterMean* __restrict__ mc, FilterShape sh,
    const int* __restrict__ perm, float4* __restrict__ full, float4* __restrict__ pre,
    double* __restrict__ place, ushort* __restrict__ extra) {
  const int64_t f = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (f >= rows) return;
  const int nseg = sh.u1 ? 2 : 1;
  if (f >= n) {  // padding: always past every threshold
    if (lane == 0) {
      full[f] = make_float4(1e30f, 0.f, 0.f, 0.f);
      pre[f] = make_float4(1e30f, 0.f, 0.f, 0.f);
    }
    for (int e = lane; e < nseg * 18; e += 64) extra[f * nseg * 18 + e] = 0;
    return;
  }
  const int64_t src = perm ? (int64_t)perm[f] : f;
  const F3* x = reinterpret_cast<const F3*>(xyz) + src * (int64_t)natoms;
  double c[3] = {0, 0, 0}, S[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  for (int i = lane; i < natoms; i += 64) {
    const F3 v = x[i];
    const double a[3] = {v.x, v.y, v.z}, wi = w[i], si = sw[i];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      c[k] += wi * a[k];
#pragma unroll
      for (int l = 0; l < 3; ++l) S[3 * k + l] += si * a[k] * mean[3 * i + l];
    }
  }
  // sum sqrt(w) m is zero up to rounding, so the uncentred sums serve: an
  // error here only turns the frame a little differently
#pragma unroll
  for (int k = 0; k < 3; ++k) c[k] = wave_sum_d(c[k]) / W;
#pragma unroll
  for (int k = 0; k < 9; ++k) S[k] = wave_sum_d(S[k]);
  double R[9];
  superpose(S, R);
  double g[2] = {0, 0}, d2[2] = {0, 0}, h2[2] = {0, 0}, l2[2] = {0, 0};
  double P[2][9] = {};
  for (int i = lane; i < natoms; i += 64) {
    const F3 v = x[i];
    const int seg = (sh.u1 && !in_first(i, sh.n0, natoms)) ? 1 : 0;
    double o[3];
    rotate3(R, (double)v.x - c[0], (double)v.y - c[1], (double)v.z - c[2], o);
    double gi = 0, di = 0, hi = 0, li = 0, d[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const double xk = (double)sw[i] * o[k];
      d[k] = xk - mean[3 * i + k];
      const double h = bf16_val(bf16_rne((float)d[k]));
      gi += xk * xk;
      di += d[k] * d[k];
      hi += h * h;
      li += (d[k] - h) * (d[k] - h);
    }
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const double on = s == seg ? 1.0 : 0.0;
      g[s] += on * gi;
      d2[s] += on * di;
      h2[s] += on * hi;
      l2[s] += on * li;
#pragma unroll
      for (int k = 0; k < 9; ++k) P[s][k] += on * d[k / 3] * mean[3 * i + k % 3];
    }
  }
  double res[2] = {0, 0};
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    if (s >= nseg) break;
    g[s] = wave_sum_d(g[s]);
    d2[s] = wave_sum_d(d2[s]);
    h2[s] = wave_sum_d(h2[s]);
    l2[s] = wave_sum_d(l2[s]);
#pragma unroll
    for (int k = 0; k < 9; ++k) {
      const double p = wave_sum_d(P[s][k]);
      const ushort ph = bf16_rne((float)p);
      const ushort pl = bf16_rne((float)(p - bf16_val(ph)));
      const double rho = p - bf16_val(ph) - bf16_val(pl);
      res[s] += rho * rho;
      if (lane == 0) {
        extra[(f * nseg + s) * 18 + k] = ph;
        extra[(f * nseg + s) * 18 + 9 + k] = pl;
      }
    }
    res[s] = 1.7320508075688772 * sqrt(res[s]);
  }
  if (lane == 0) {
    const double up = 1.0 + 1e-6;
    const double gt = g[0] + g[1];
    const double dn0 = sqrt(fmax(d2[0], h2[0])), dn = sqrt(fmax(d2[0] + d2[1], h2[0] + h2[1]));
    const double step = 5.2 * 2.384185791015625e-7;  // 5.2 x 2^-22
    const double a0 = mc->norm0 + dn0, a = mc->norm + dn;
    const double e0 = step * (sh.groups0() + 2) * 0.5 * a0 * a0;
    const double e1 = step * (sh.groups() + 4) * 0.5 * a * a;
    // A frame whose squares leave FP32's range (or that is not finite) is
    // never past a threshold: every comparison with NaN keeps its tiles.  The
    // test's square roots take squares below 1.2e-38 as zero, so that its sum
    // of column norms may be short by 3.3e-19: from 1e-12 on that is less than
    // the 1e-6 gt taken off below.
    const double nan = gt >= 1e-12 && gt <= 1e29 ? 0.0 : (double)NAN;
    full[f] = make_float4((float)(0.5 * gt - res[0] - res[1] - e1 - 1e-6 * gt + nan),
                          (float)(dn * up), (float)(sqrt(l2[0] + l2[1]) * up), 0.f);
    pre[f] = make_float4((float)(0.5 * gt - res[0] - e0 - 1e-6 * gt + nan), (float)(dn0 * up),
                         (float)(sqrt(l2[0]) * up), (float)(sqrt(g[1]) * up));
  }
  if (lane < 12) place[f * 12 + lane] = lane < 9 ? R[lane] : c[lane - 9];
}

constexpr int kOpGroups = 4;  // K-groups per operand workgroup (divides every segment)

// The operand in fragment order: one workgroup per (tile, 4 K-groups),
// thread t on plane t/64, lane t%64.  The last K-group of a segment holds
// its extra slots and exists twice: in place for the reference side, and at
// K-group groups() + segment for the fit side.
__global__ __launch_bounds__(192) void filter_operand_kernel(
    const float* __restrict__ xyz, int64_t n, int natoms, const float* __restrict__ sw,
    const double* __restrict__ mean, FilterShape sh, const int* __restrict__ slots,
    const int* __restrict__ perm, const double* __restrict__ place,
    const ushort* __restrict__ extra, uint4* __restrict__ op) {
  constexpr int kSlots = 16 * kOpGroups;
  constexpr int kPitch = 3 * kSlots + 1;
  __shared__ float xs[kTile * kPitch];
  __shared__ int sslot[kSlots];
  const int tile = blockIdx.x, g0 = blockIdx.y * kOpGroups, t = threadIdx.x;
  const int nseg = sh.u1 ? 2 : 1;
  if (t < kSlots) sslot[t] = slots[g0 * 16 + t];
  __syncthreads();
  for (int i = t; i < kTile * kSlots; i += 192) {
    const int fr = i / kSlots, s = i - fr * kSlots;
    const int64_t ff = (int64_t)tile * kTile + fr;
    const int a = sslot[s];
    F3 v = {0.f, 0.f, 0.f};
    if (ff < n && a >= 0)
      v = (reinterpret_cast<const F3*>(xyz) + (perm ? (int64_t)perm[ff] : ff) * natoms)[a];
    xs[fr * kPitch + 3 * s] = v.x;
    xs[fr * kPitch + 3 * s + 1] = v.y;
    xs[fr * kPitch + 3 * s + 2] = v.z;
  }
  __syncthreads();
  const int c = t >> 6, lane = t & 63, row = lane & 31, h = lane >> 5;
  const int64_t f = (int64_t)tile * kTile + row;
  double R0 = 0, R1 = 0, R2 = 0, c0 = 0, c1 = 0, c2 = 0;
  if (f < n) {
    const double* p = place + f * 12;
    R0 = p[3 * c]; R1 = p[3 * c + 1]; R2 = p[3 * c + 2];
    c0 = p[9]; c1 = p[10]; c2 = p[11];
  }
  const int64_t tile_groups = sh.groups() + nseg;
#pragma unroll
  for (int gg = 0; gg < kOpGroups; ++gg) {
    const int g = g0 + gg;
    const int seg = (sh.u1 && g >= sh.groups0()) ? 1 : 0;
    const bool last = g == (seg ? sh.groups() : sh.groups0()) - 1;
    ushort ref[8], fit[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int s = gg * 16 + 8 * h + j;
      const int a = sslot[s];
      ushort r = 0, q = 0;
      if (f < n) {
        if (a >= 0) {
          const float* xr = xs + row * kPitch + 3 * s;
          const double o = fma(R2, (double)xr[2] - c2, fma(R1, (double)xr[1] - c1,
                                                          R0 * ((double)xr[0] - c0)));
          r = q = bf16_rne((float)((double)sw[a] * o - mean[3 * a + c]));
        } else if (a <= -2) {
          const int e = -2 - a, col = e % 3;
          const ushort* p = extra + (f * nseg + seg) * 18 + (e / 3 & 1) * 9 + 3 * c + col;
          const ushort unit = col == c ? 0x3F80 : 0;  // 1.0
          r = e < 6 ? *p : unit;
          q = e < 6 ? unit : *p;
        }
      }
      ref[j] = r;
      fit[j] = q;
    }
    auto pack = [](const ushort* v) {
      uint4 o;
      o.x = v[0] | ((unsigned)v[1] << 16); o.y = v[2] | ((unsigned)v[3] << 16);
      o.z = v[4] | ((unsigned)v[5] << 16); o.w = v[6] | ((unsigned)v[7] << 16);
      return o;
    };
    op[((tile * tile_groups + g) * 3 + c) * 64 + lane] = pack(ref);
    if (last) op[((tile * tile_groups + sh.groups() + seg) * 3 + c) * 64 + lane] = pack(fit);
  }
}

// ---------------------------------------------------------------------------
// the filter

// Waits for this wave's LDS reads (and, N >= 0, its copies but the last N),
// then the workgroup barrier.
template <int N>
__device__ __forceinline__ void fence_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4));
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}
// The K-loop's stage end: copies older than the last N landed; LDS reads
// stay in flight (they are of a buffer no copy touches before the next one).
template <int N>
__device__ __forceinline__ void stage_end() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4) | (0xF << 8));
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

__device__ __forceinline__ void mma3(f32x16 (&acc)[9], int c, const uint4 a, const uint4 (&b)[3]) {
#pragma unroll
  for (int d = 0; d < 3; ++d)
    acc[c * 3 + d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
        __builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b[d]), acc[c * 3 + d], 0, 0, 0);
}

// One K-group from the current buffer (plane 0's A and the three B already
// in registers), reading the next group's B and plane-0 A as it goes.
__device__ __forceinline__ void group_step(f32x16 (&acc)[9], const uint4* __restrict__ ca,
                                           const uint4* __restrict__ na,
                                           const uint4* __restrict__ nb, const uint4 (&b)[3],
                                           uint4 (&bn)[3], uint4& a, int lane) {
  const uint4 a1 = ca[64 + lane];
  bn[0] = nb[lane];
  mma3(acc, 0, a, b);
  const uint4 a2 = ca[128 + lane];
  bn[1] = nb[64 + lane];
  mma3(acc, 1, a1, b);
  a = na[lane];
  bn[2] = nb[128 + lane];
  mma3(acc, 2, a2, b);
}

// One stage: GPS K-groups.  b holds the stage's first group's B on entry and
// (GPS 2) the next stage's on exit; with GPS 1 the next stage's is in bn.
template <int GPS>
__device__ __forceinline__ void stage_step(f32x16 (&acc)[9], const uint4* __restrict__ ca,
                                           const uint4* __restrict__ cb,
                                           const uint4* __restrict__ na,
                                           const uint4* __restrict__ nb, uint4 (&b)[3],
                                           uint4 (&bn)[3], uint4& a, int lane) {
  if constexpr (GPS == 1) {
    group_step(acc, ca, na, nb, b, bn, a, lane);
  } else {
    group_step(acc, ca, ca + 192, cb + 192, b, bn, a, lane);
    group_step(acc, ca + 192, na, nb, bn, b, a, lane);
  }
}

struct FilterParams {
  const uint4* rop;
  const uint4* fop;
  const float4* rfull;
  const float4* rpre;
  const float4* ffull;
  const float4* fpre;
  const FilterMean* mc;
  FilterShape sh;
  int64_t n_ref, n_fit;
  int ref_pairs, fit_blocks, phases;
  const unsigned* thr;
  const float* eps2;
  // the reference pairs to test, per fit block (rows of ref_pairs entries)
  const int* list;
  const int* count;
  unsigned char* flags;
  const int* ctrl;
  int part;
};

constexpr int kSampleEvery = 16;

// The fit blocks of one part of the filter: every kSampleEvery-th block
// (part 0, the sample that decides whether the rest is worth it), the others
// (part 1), or all of them (part 2, few blocks).
__host__ __device__ __forceinline__ int part_blocks(int fit_blocks, int part) {
  const int s = (fit_blocks + kSampleEvery - 1) / kSampleEvery;
  return part == 0 ? s : part == 1 ? fit_blocks - s : fit_blocks;
}
__device__ __forceinline__ int part_block(int i, int part) {
  return part == 0 ? i * kSampleEvery : part == 1 ? i + i / (kSampleEvery - 1) + 1 : i;
}

// Too many tiles of the sample are left: the contraction takes every tile.
__device__ __forceinline__ bool not_worth(const int* ctrl) {
  return (int64_t)ctrl[0] * 100 > (int64_t)ctrl[1] * 60;
}

// Persistent, one 8-wave workgroup per CU; item (fit block of 4 tiles,
// phase), wave = one 32 x 32 tile, the contraction's geometry and pipeline
// (four LDS stage buffers, copies three stages ahead, fragments read one
// group ahead).  SYM: a self query, reference pairs from the block's own
// first frame on, and a pair must be past both frames' thresholds.
// Bound by the LDS reads (6 KiB per wave and K-group for 9 MFMAs, 288
// cycles) and the matrix cores; the bound's test takes about 20 FP32
// instructions and 3 square roots per pair.
template <int GPS, bool SYM>
__global__ __launch_bounds__(512, 2) void filter_kernel(FilterParams P) {
  constexpr int FT = 4;
  constexpr int BPG = 3 * GPS;
  constexpr int TILE_VEC = BPG * 64;
  constexpr int STAGE_VEC = (kRefTilesPerWG + FT) * TILE_VEC;
  constexpr int kSlots = kRefTilesPerWG + FT;
  __shared__ uint4 sbuf0[STAGE_VEC];
  __shared__ uint4 sbuf1[STAGE_VEC];
  __shared__ uint4 sbuf2[STAGE_VEC];
  __shared__ uint4 sbuf3[STAGE_VEC];
  __shared__ float4 sRow[2][2][2 * kTile];  // [tile parity][first segment only / all]
  __shared__ float sT[2][2 * kTile];
  __shared__ int sVote[2][8];

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int ri = wave & 1, fi = wave >> 1;
  const bool copier = wave < kSlots;
  const int slot = copier ? wave : 0;
  uint4* const d0 = sbuf0 + slot * TILE_VEC;
  uint4* const d1 = sbuf1 + slot * TILE_VEC;
  uint4* const d2 = sbuf2 + slot * TILE_VEC;
  uint4* const d3 = sbuf3 + slot * TILE_VEC;
  const uint4* const a0 = sbuf0 + ri * TILE_VEC;
  const uint4* const a1 = sbuf1 + ri * TILE_VEC;
  const uint4* const a2 = sbuf2 + ri * TILE_VEC;
  const uint4* const a3 = sbuf3 + ri * TILE_VEC;
  const uint4* const b0 = sbuf0 + (kRefTilesPerWG + fi) * TILE_VEC;
  const uint4* const b1 = sbuf1 + (kRefTilesPerWG + fi) * TILE_VEC;
  const uint4* const b2 = sbuf2 + (kRefTilesPerWG + fi) * TILE_VEC;
  const uint4* const b3 = sbuf3 + (kRefTilesPerWG + fi) * TILE_VEC;

  const int nseg = P.sh.u1 ? 2 : 1;
  const int ns0 = 4 * P.sh.u0, ns = 4 * (P.sh.u0 + P.sh.u1);
  const int64_t tile_vec = (int64_t)(P.sh.groups() + nseg) * 192;
  const bool skip = P.part == 1 && not_worth(P.ctrl);

  const int nwg = gridDim.x;
  const int logical = (int)(blockIdx.x & 7) * (nwg >> 3) + (int)(blockIdx.x >> 3);
  const int n_items = part_blocks(P.fit_blocks, P.part) * P.phases;

  auto threshold = [&](int64_t f, int64_t n) -> float {
    // half the row's threshold, with its window's half on top
    return f < n ? 0.5f * (__uint_as_float(P.thr[f]) + 0.5f * P.eps2[f]) * (1.0f + 1e-6f) : 0.f;
  };

  for (int item = logical; item < n_items; item += nwg) {
    const int bi = item / P.phases;
    const int ph = item - bi * P.phases;
    const int fb = part_block(bi, P.part);
    const int n_tiles = (P.count[fb] - ph + P.phases - 1) / P.phases;
    if (n_tiles <= 0) continue;
    const int* const list = P.list + (int64_t)fb * P.ref_pairs + ph;
    unsigned char* const flags = P.flags + (int64_t)fb * P.ref_pairs;
    if (skip) {
      for (int t = tid; t < n_tiles; t += 512) flags[list[t * P.phases]] = 1;
      continue;
    }
    auto pair_of = [&](int t) -> int {
      return __builtin_amdgcn_readfirstlane(list[min(t, n_tiles - 1) * P.phases]);
    };
    int p = pair_of(0), p_next = pair_of(1);
    const int64_t fit_idx = (int64_t)(FT * fb + fi) * kTile + (lane & 31);
    const float4 ff = P.ffull[fit_idx], fp = P.fpre[fit_idx];
    const float tf = threshold(fit_idx, P.n_fit);
    // Test after the first segment?  After the n-th miss in a row the next
    // 2^n tiles (up to 64) take both segments at once: the tiles next to the
    // block are all kept, and a set the first segment cannot split costs
    // little.
    bool two = nseg == 2;
    int misses = 0, hold = 0;

    const uint4* const fit_base = P.fop + (int64_t)(FT * fb + slot - kRefTilesPerWG) * tile_vec;
    // stage s of reference pair q
    auto dma = [&](int q, int s, uint4* dst) {
      if (!copier) return;
      const bool ref = wave < kRefTilesPerWG;
      const uint4* const base =
          ref ? P.rop + (int64_t)(kRefTilesPerWG * q + wave) * tile_vec : fit_base;
#pragma unroll
      for (int u = 0; u < GPS; ++u) {
        int g = s * GPS + u;
        // the fit side's copy of a segment's last K-group
        if (!ref && u == GPS - 1) {
          if (s == ns0 - 1) g = ns * GPS;
          else if (s == ns - 1) g = ns * GPS + 1;
        }
        const uint4* const src = base + g * 192 + lane;
#pragma unroll
        for (int j = 0; j < 3; ++j)
          __builtin_amdgcn_global_load_lds((const void*)(src + j * 64),
                                           (lds_void_t*)(dst + (u * 3 + j) * 64), 16, 0, 0);
      }
    };

    __syncthreads();  // previous item's readers are done
    if (tid < 2 * kTile) {
      const int64_t f0 = (int64_t)p * 2 * kTile + tid;
      sRow[0][0][tid] = P.rpre[f0];
      sRow[0][1][tid] = P.rfull[f0];
      sT[0][tid] = SYM ? threshold(f0, P.n_ref) : -FLT_MAX;
    }
    dma(p, 0, d0);
    dma(p, 1, d1);
    dma(p, 2, d2);
    fence_barrier<BPG>();
    uint4 bA[3], bB[3], a;
#pragma unroll
    for (int d = 0; d < 3; ++d) bA[d] = b0[d * 64 + lane];
    a = a0[lane];

    for (int t = 0; t < n_tiles; ++t) {
      float4 next_pre = make_float4(0, 0, 0, 0), next_full = make_float4(0, 0, 0, 0);
      float next_t = -FLT_MAX;
      if (tid < 2 * kTile && t + 1 < n_tiles) {
        const int64_t f1 = (int64_t)p_next * 2 * kTile + tid;
        next_pre = P.rpre[f1];
        next_full = P.rfull[f1];
        if constexpr (SYM) next_t = threshold(f1, P.n_ref);
      }
      f32x16 acc[9];
#pragma unroll
      for (int q = 0; q < 9; ++q) {
        const float cq = P.mc->C[0][q] + (two ? 0.f : P.mc->C[1][q]);
        acc[q] = (f32x16){cq, cq, cq, cq, cq, cq, cq, cq, cq, cq, cq, cq, cq, cq, cq, cq};
      }
      // Stages s0 .. s1-1 of tile t; the copies run three stages ahead, past s1
      // into the next tile.
      auto run = [&](int s0, int s1) {
        for (int s = s0; s < s1; s += 4) {
          const bool more = s + 4 < s1;
          const int pn = more ? p : p_next, sn = more ? s + 4 : 0;
          stage_step<GPS>(acc, a0, b0, a1, b1, bA, bB, a, lane);
          dma(p, s + 3, d3);
          stage_end<BPG>();
          stage_step<GPS>(acc, a1, b1, a2, b2, GPS == 1 ? bB : bA, GPS == 1 ? bA : bB, a, lane);
          dma(pn, sn, d0);
          stage_end<BPG>();
          stage_step<GPS>(acc, a2, b2, a3, b3, bA, bB, a, lane);
          dma(pn, sn + 1, d1);
          stage_end<BPG>();
          stage_step<GPS>(acc, a3, b3, a0, b0, GPS == 1 ? bB : bA, GPS == 1 ? bA : bB, a, lane);
          dma(pn, sn + 2, d2);
          stage_end<BPG>();
        }
      };
      // Whether a pair of this wave may lie below a threshold: lane = fit
      // frame, 16 reference frames.
      auto test = [&](const float4* __restrict__ rows, const float4 fk) -> bool {
        const float4* const row = rows + ri * kTile;
        const float* const rt = sT[t & 1] + ri * kTile;
        bool alive = false;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int rl = 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
          const float4 k = row[rl];
          float lub = 0.f;
#pragma unroll
          for (int d = 0; d < 3; ++d)
            lub += __builtin_amdgcn_sqrtf(fmaf(acc[d][r], acc[d][r],
                                               fmaf(acc[3 + d][r], acc[3 + d][r],
                                                    acc[6 + d][r] * acc[6 + d][r])));
          float lim = k.x + fk.x - fmaxf(rt[rl], tf) - fmaf(fk.y, k.z, fmaf(fk.z, k.y, fk.w * k.w));
          // opaque: the rows are otherwise joined into 16-wide vectors whose
          // splats of fk are kept (spilled) across the tile loop
          asm volatile("" : "+v"(lub), "+v"(lim));
          alive |= !(lub * (1.0f + 3e-6f) < lim);
        }
        return __any(alive);
      };
      run(0, two ? ns0 : ns);
      bool second = !two;
      bool wave_alive = test(sRow[t & 1][second ? 1 : 0], second ? ff : fp);
      if (two) {
        // does any wave need the second segment?
        if (lane == 0) sVote[t & 1][wave] = wave_alive;
        fence_barrier<63>();
        int any = 0;
#pragma unroll
        for (int v = 0; v < 8; ++v) any |= sVote[t & 1][v];
        any = __builtin_amdgcn_readfirstlane(any);
        if (!any) misses = 0;
        if (any) {
          misses = min(misses + 1, 6);
          hold = 1 << misses;
          second = true;
          // the buffers hold the next tile's first stages: fill them again
          // with this tile's second segment
          fence_barrier<0>();
          dma(p, ns0, d0);
          dma(p, ns0 + 1, d1);
          dma(p, ns0 + 2, d2);
#pragma unroll
          for (int q = 0; q < 9; ++q) {
            const float cq = P.mc->C[1][q];
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[q][r] += cq;
          }
          fence_barrier<BPG>();
#pragma unroll
          for (int d = 0; d < 3; ++d) bA[d] = b0[d * 64 + lane];
          a = a0[lane];
          run(ns0, ns);
          wave_alive = test(sRow[t & 1][1], ff);
        }
      }
      if (second && wave_alive && lane == 0) flags[p] = 1;
      if (hold > 0) --hold;
      two = nseg == 2 && hold == 0;
      if (tid < 2 * kTile && t + 1 < n_tiles) {
        sRow[(t + 1) & 1][0][tid] = next_pre;
        sRow[(t + 1) & 1][1][tid] = next_full;
        sT[(t + 1) & 1][tid] = next_t;
      }
      p = p_next;
      p_next = pair_of(t + 2);
    }
  }
}

// The middle frame of each 64 (the frames of a reference pair): its index
// among the frames as given.
__global__ void middle_kernel(const int* __restrict__ order, int64_t n, int groups,
                              int* __restrict__ mid) {
  const int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g < groups) mid[g] = order[min((int64_t)g * 2 * kTile + kTile, n - 1)];
}

// One workgroup per fit block of a part: its flagged reference pairs in
// ascending order, in place of the tested ones; ctrl[0/1] += flagged / tested
// pairs (part 0).  flags null: all of them.
__global__ __launch_bounds__(256) void filter_list_kernel(const unsigned char* __restrict__ flags,
                                                          int ref_pairs, int fit_blocks, int part,
                                                          int sym_step, int* __restrict__ list,
                                                          int* __restrict__ count,
                                                          int* __restrict__ ctrl) {
  const int fb = part_block(blockIdx.x, part);
  if (fb >= fit_blocks) return;
  const unsigned char* const f = flags ? flags + (int64_t)fb * ref_pairs : nullptr;
  int* const out = list + (int64_t)fb * ref_pairs;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  __shared__ int part_n[4];
  const int tested = count[fb];
  int base = 0;
  for (int p0 = fb * sym_step; p0 < ref_pairs; p0 += 256) {
    const int p = p0 + tid;
    const bool on = p < ref_pairs && (!f || f[p]);
    const uint64_t b = __ballot(on);
    if (lane == 0) part_n[wave] = __popcll(b);
    __syncthreads();
    int at = base;
    for (int v = 0; v < wave; ++v) at += part_n[v];
    if (on) out[at + __popcll(b & ((1ull << lane) - 1ull))] = p;
    base += part_n[0] + part_n[1] + part_n[2] + part_n[3];
    __syncthreads();
  }
  if (tid == 0) {
    count[fb] = base;
    if (part == 0) {
      atomicAdd(&ctrl[0], base);
      atomicAdd(&ctrl[1], tested);
    }
  }
}

// The band pass's tile list: each fit block against the `width` reference
// pairs around it.
__global__ void band_list_kernel(int ref_pairs, int fit_blocks, int block_pairs, int width,
                                 int* __restrict__ list, int* __restrict__ count) {
  const int fb = blockIdx.x;
  int lo = fb * block_pairs + block_pairs / 2 - width / 2;
  lo = max(0, min(lo, ref_pairs - width));
  const int m = min(width, ref_pairs - lo);
  for (int i = threadIdx.x; i < m; i += blockDim.x) list[(int64_t)fb * ref_pairs + i] = lo + i;
  if (threadIdx.x == 0) count[fb] = m;
}

// The same for a cross query: the rows of a block are in the order of their
// keys, places in the ordered set, and may stand around several of them: the
// `width` reference pairs around each row's place.  One row without a
// candidate nearby keeps every tile of its block, so all rows count unless
// that makes more than `most` pairs; then every second, fourth ... row.
__global__ __launch_bounds__(128) void place_band_list_kernel(
    const unsigned* __restrict__ keys, int dist_bits, const int* __restrict__ order, int64_t n,
    int ref_pairs, int width, int most, int* __restrict__ list, int* __restrict__ count) {
  constexpr int kRows = kFilterFitTiles * kTile;
  __shared__ int at[kRows];
  const int fb = blockIdx.x;
  const int64_t row = min((int64_t)fb * kRows + threadIdx.x, n - 1);
  at[threadIdx.x] = (int)((keys[order[row]] >> dist_bits) / (2u * kTile));
  __syncthreads();
  if (threadIdx.x) return;
  int* const out = list + (int64_t)fb * ref_pairs;
  auto walk = [&](int step, bool write) {
    int m = 0, end = 0;
    for (int r = step / 2; r < kRows; r += step) {
      const int lo = max(max(0, min(at[r] - width / 2, ref_pairs - width)), end);
      const int hi = min(max(0, min(at[r] - width / 2, ref_pairs - width)) + width, ref_pairs);
      if (write)
        for (int p = lo; p < hi; ++p) out[m + p - lo] = p;
      m += max(0, hi - lo);
      end = max(end, hi);
    }
    return m;
  };
  int step = 1;
  while (step < kRows / 4 && walk(step, false) > most) step *= 2;
  count[fb] = walk(step, true);
}

__global__ void clear_kernel(uint4* p, int64_t n, int* ctrl) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = make_uint4(0, 0, 0, 0);
  if (i < 2 && ctrl) ctrl[i] = 0;
}

// The last of a cell's chain of leaders (each leader is the cell itself or an
// earlier one, so the chain ends).
__device__ __forceinline__ int chief(const int* __restrict__ leaders, int c) {
  for (int l = leaders[c]; l >= 0 && l < c; l = leaders[c]) c = l;
  return c;
}

// A cell's place when cells are sorted by (chief, cell).
__global__ __launch_bounds__(256) void cell_rank_kernel(const int* __restrict__ leaders, int ncells,
                                                        int* __restrict__ rank) {
  const int c = blockIdx.x * 256 + threadIdx.x;
  const int mine = c < ncells ? chief(leaders, c) : 0;
  __shared__ int other[256];
  int r = 0;
  for (int j0 = 0; j0 < ncells; j0 += 256) {
    __syncthreads();
    other[threadIdx.x] =
        j0 + (int)threadIdx.x < ncells ? chief(leaders, j0 + (int)threadIdx.x) : INT_MAX;
    __syncthreads();
    for (int j = 0; j < 256; ++j)
      r += other[j] < mine || (other[j] == mine && j0 + j < c);
  }
  if (c < ncells) rank[c] = r;
}

__global__ void fill_near_kernel(unsigned long long* p, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = ~0ull;
}

// A frame's cell is its nearest landmark (numbered densely, as
// landmark_cap_kernel does), then its distance's leading bits.
__global__ void near_keys_kernel(const unsigned long long* __restrict__ near, int64_t n, int phases,
                                 unsigned* __restrict__ keys, int* __restrict__ rows) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= n) return;
  const unsigned long long b = near[q];
  const unsigned r = (unsigned)b, span = 2u * kTile * (unsigned)phases;
  const unsigned cell = b == ~0ull ? 0u : (r / span) * (2u * kTile) + r % (2u * kTile);
  keys[q] = (cell << kFilterDistBits) |
            ((unsigned)(b >> 32) >> (31 - kFilterDistBits) & ((1u << kFilterDistBits) - 1u));
  rows[q] = (int)q;
}

__global__ void places_kernel(const int* __restrict__ order, int64_t n, int* __restrict__ place) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) place[order[i]] = (int)i;
}

// order[place of row q among the keys] = q: 64 rows a workgroup against all
// keys, a quarter of them per wave, four per LDS read.
__global__ __launch_bounds__(256) void rank_sort_kernel(const unsigned* __restrict__ keys, int n,
                                                        int* __restrict__ order) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int q = blockIdx.x * 64 + lane;
  const unsigned mine = q < n ? keys[q] : 0u;
  __shared__ __align__(16) unsigned other[1024];
  __shared__ int part[4][64];
  int r = 0;
  for (int j0 = 0; j0 < n; j0 += 1024) {
    __syncthreads();
    for (int j = threadIdx.x; j < 1024; j += 256) other[j] = j0 + j < n ? keys[j0 + j] : 0xffffffffu;
    __syncthreads();
    const uint4* const o = reinterpret_cast<const uint4*>(other) + wave * 64;
    const int base = j0 + wave * 256;
    // keys past n compare as larger, and none of them equals a key below q
#pragma unroll 4
    for (int j = 0; j < 64; ++j) {
      const uint4 k = o[j];
      const int at = base + 4 * j;
      r += k.x < mine || (k.x == mine && at < q);
      r += k.y < mine || (k.y == mine && at + 1 < q);
      r += k.z < mine || (k.z == mine && at + 2 < q);
      r += k.w < mine || (k.w == mine && at + 3 < q);
    }
  }
  part[wave][lane] = r;
  __syncthreads();
  if (wave == 0 && q < n) order[part[0][lane] + part[1][lane] + part[2][lane] + part[3][lane]] = q;
}

// One pass of the stable sort by digits of 8 bits, in two kernels of at most
// kSortBlocks workgroups of 4 waves.  A wave takes 64 rows a round, `rounds`
// rounds side by side, so rows keep their order within a digit: workgroups,
// waves, rounds, lanes.  Bound by its eight launches and each pass's chain of
// loads: 5000 rows 26 us, 40007 35, 200000 72, 1000000 123.  (hipCUB's sort took
// 24, 38, 60 and 164, and its 468 kernels 4 ms to load on a process's first use.)
constexpr int kSortBlocks = 256;

// counts[workgroup][digit] of the rows of each workgroup.
__global__ __launch_bounds__(256) void sort_count_kernel(const unsigned* __restrict__ keys, int n,
                                                         int rounds, int shift,
                                                         int* __restrict__ counts) {
  __shared__ int bin[256];
  const int tid = threadIdx.x;
  bin[tid] = 0;
  __syncthreads();
  const int64_t i0 = (int64_t)blockIdx.x * rounds * 256 + tid;
  for (int r = 0; r < rounds; r += 4) {
    unsigned k[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int64_t i = i0 + (r + j) * 256;
      k[j] = i < n ? keys[i] : 0u;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (i0 + (r + j) * 256 < n) atomicAdd(&bin[k[j] >> shift & 255u], 1);
  }
  __syncthreads();
  counts[blockIdx.x * 256 + tid] = bin[tid];
}

// Rows to their places by that digit.  A digit's rows start after all rows of
// smaller digits and those of the workgroups and waves before; within a wave's
// round a lane's place is the number of lower lanes with its digit.
__global__ __launch_bounds__(256) void sort_scatter_kernel(
    const unsigned* __restrict__ keys, const int* __restrict__ rows, int n, int rounds, int shift,
    const int* __restrict__ counts, unsigned* __restrict__ keys_out, int* __restrict__ rows_out) {
  __shared__ int at[4][256];
  __shared__ int wave_sum[4];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  for (int w = 0; w < 4; ++w) at[w][tid] = 0;
  __syncthreads();
  const int64_t i0 = ((int64_t)blockIdx.x * 4 + wave) * rounds * 64 + lane;
  unsigned k[4];
  auto load = [&](int r) {  // the keys of four rounds
#pragma unroll
    for (int j = 0; j < 4; ++j) k[j] = i0 + (r + j) * 64 < n ? keys[i0 + (r + j) * 64] : 0u;
  };
  for (int r = 0; r < rounds; r += 4) {
    load(r);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (i0 + (r + j) * 64 < n) atomicAdd(&at[wave][k[j] >> shift & 255u], 1);
  }
  // thread = digit: its rows in all workgroups, and in those before this one
  // (sixteen loads in flight: one by one, 200000 rows took 208 us)
  int total = 0, before = 0;
  for (int b0 = 0; b0 < (int)gridDim.x; b0 += 16) {
    int c[16];
#pragma unroll
    for (int j = 0; j < 16; ++j)
      c[j] = b0 + j < (int)gridDim.x ? counts[(b0 + j) * 256 + tid] : 0;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      total += c[j];
      before += b0 + j < (int)blockIdx.x ? c[j] : 0;
    }
  }
  int upto = total;  // inclusive sum over the digits
  for (int o = 1; o < 64; o <<= 1) {
    const int v = __shfl_up(upto, o);
    upto += lane >= o ? v : 0;
  }
  if (lane == 63) wave_sum[wave] = upto;
  __syncthreads();
  int start = before + upto - total;
  for (int w = 0; w < wave; ++w) start += wave_sum[w];
  for (int w = 0; w < 4; ++w) {
    const int c = at[w][tid];
    at[w][tid] = start;
    start += c;
  }
  __syncthreads();
  for (int r = 0; r < rounds; r += 4) {
    if (rounds > 4) load(r);  // else they are the ones counted
    int row[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) row[j] = i0 + (r + j) * 64 < n ? rows[i0 + (r + j) * 64] : 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const bool on = i0 + (r + j) * 64 < n;
      const unsigned digit = k[j] >> shift & 255u;
      uint64_t same = __ballot(on);
#pragma unroll
      for (int bit = 0; bit < 8; ++bit) {
        const uint64_t set = __ballot(digit >> bit & 1u);
        same &= digit >> bit & 1u ? set : ~set;
      }
      const int rank = __popcll(same & ((1ull << lane) - 1ull));
      // the first lane of a digit takes the places of all its lanes
      int base = 0;
      if (on && rank == 0) base = atomicAdd(&at[wave][digit], __popcll(same));
      base = __shfl(base, on ? __builtin_ctzll(same) : lane);
      if (on) {
        keys_out[base + rank] = k[j];
        rows_out[base + rank] = row[j];
      }
    }
  }
}

__global__ void rank_keys_kernel(const int* __restrict__ rank, int ncells, int64_t n,
                                 unsigned* __restrict__ keys) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= n) return;
  const unsigned k = keys[q], c = k >> kFilterDistBits;
  keys[q] = ((unsigned)rank[min((int)c, ncells - 1)] << kFilterDistBits) |
            (k & ((1u << kFilterDistBits) - 1u));
}

}  // namespace

FilterShape filter_shape(int natoms) {
  FilterShape s;
  s.natoms = natoms;
  // two K-groups per stage from 384 slots on (deeper prefetch), one below
  // (less padding)
  s.gps = natoms + kFilterExtra > 320 ? 2 : 1;
  const int unit = 64 * s.gps;
  if (natoms >= 384) {
    s.u0 = std::max(1, (natoms / 4 + kFilterExtra + unit / 2) / unit);
    s.n0 = s.u0 * unit - kFilterExtra;
    s.u1 = (natoms - s.n0 + kFilterExtra + unit - 1) / unit;
  } else {
    s.u0 = (natoms + kFilterExtra + unit - 1) / unit;
    s.n0 = natoms;
    s.u1 = 0;
  }
  return s;
}

size_t filter_operand_bytes(const FilterShape& s, int n_tiles) {
  return (size_t)n_tiles * (s.groups() + (s.u1 ? 2 : 1)) * 3 * 64 * 16;
}

hipError_t launch_filter_mean(const DevFrames& f, const DevWeights& w, const FilterShape& sh,
                              double* scratch, double* mean, FilterMean* mc, int* slots,
                              hipStream_t st) {
  const int samples = (int)std::min<int64_t>(kFilterSamples, f.n);
  hipLaunchKernelGGL(mean_align_kernel, dim3((samples + 3) / 4), dim3(256), 0, st, f.xyz, f.n,
                     f.natoms, w.w, w.W, samples, scratch);
  hipLaunchKernelGGL(mean_sum_kernel, dim3((f.natoms + 63) / 64), dim3(64), 0, st, f.xyz, f.n,
                     f.natoms, samples, scratch, mean);
  hipLaunchKernelGGL(mean_final_kernel, dim3(1), dim3(256), 0, st, w.w, w.sw, f.natoms, sh, mean,
                     mc, slots);
  return hipGetLastError();
}

hipError_t launch_filter_prep(const DevFrames& f, const DevWeights& w, const FilterShape& sh,
                              const double* mean, const FilterMean* mc, const int* slots,
                              const int* perm, const FilterSet& out, hipStream_t st) {
  const int64_t rows = (int64_t)f.n_tiles * kTile;
  hipLaunchKernelGGL(filter_stats_kernel, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, st, f.xyz,
                     f.n, rows, f.natoms, w.w, w.sw, w.W, mean, mc, sh, perm, out.full, out.pre,
                     out.place, out.extra);
  hipLaunchKernelGGL(filter_operand_kernel,
                     dim3((unsigned)f.n_tiles, (unsigned)(sh.groups() / kOpGroups)), dim3(192), 0,
                     st, f.xyz, f.n, f.natoms, w.sw, mean, sh, slots, perm, out.place, out.extra,
                     out.op);
  return hipGetLastError();
}

hipError_t launch_filter(const FilterSet& ref, const FilterSet& fit, int64_t n_ref, int64_t n_fit,
                         int ref_tiles, int fit_tiles, const FilterShape& sh, const FilterMean* mc,
                         const unsigned* thr, const float* eps2, bool sym, int grid,
                         const TileList& tl, const unsigned char* test, hipStream_t st) {
  constexpr int FT = 4;
  FilterParams P;
  P.rop = ref.op;
  P.fop = fit.op;
  P.rfull = ref.full;
  P.rpre = ref.pre;
  P.ffull = fit.full;
  P.fpre = fit.pre;
  P.mc = mc;
  P.sh = sh;
  P.n_ref = n_ref;
  P.n_fit = n_fit;
  P.ref_pairs = ref_tiles / kRefTilesPerWG;
  P.fit_blocks = fit_tiles / FT;
  P.thr = thr;
  P.eps2 = eps2;
  P.list = tl.list;
  P.count = tl.count;
  P.flags = tl.flags;
  P.ctrl = tl.ctrl;
  if (ref_tiles % kRefTilesPerWG || fit_tiles % FT || grid < 8 || (grid & 7))
    return hipErrorInvalidValue;
  const int64_t vec = ((int64_t)P.fit_blocks * P.ref_pairs + 15) / 16;
  hipLaunchKernelGGL(clear_kernel, dim3((unsigned)((vec + 255) / 256)), dim3(256), 0, st,
                     reinterpret_cast<uint4*>(tl.flags), vec, tl.ctrl);
  hipLaunchKernelGGL(filter_list_kernel, dim3((unsigned)P.fit_blocks), dim3(256), 0, st, test,
                     P.ref_pairs, P.fit_blocks, 2, sym ? FT / kRefTilesPerWG : 0, tl.list, tl.count,
                     tl.ctrl);
  // The sample costs two launches: from 64 blocks on.  Phases so that every
  // workgroup gets about four items, of eight tiles or more.
  for (int part = P.fit_blocks >= 64 ? 0 : 2; part < 3; part += part == 1 ? 2 : 1) {
    const int blocks = part_blocks(P.fit_blocks, part);
    P.part = part;
    P.phases = 4;
    while (P.phases * blocks < 4 * grid && P.phases * 16 <= P.ref_pairs) P.phases *= 2;
    if (sh.gps == 1) {
      if (sym)
        hipLaunchKernelGGL((filter_kernel<1, true>), dim3(grid), dim3(512), 0, st, P);
      else
        hipLaunchKernelGGL((filter_kernel<1, false>), dim3(grid), dim3(512), 0, st, P);
    } else {
      if (sym)
        hipLaunchKernelGGL((filter_kernel<2, true>), dim3(grid), dim3(512), 0, st, P);
      else
        hipLaunchKernelGGL((filter_kernel<2, false>), dim3(grid), dim3(512), 0, st, P);
    }
    hipLaunchKernelGGL(filter_list_kernel, dim3((unsigned)blocks), dim3(256), 0, st, tl.flags,
                       P.ref_pairs, P.fit_blocks, part, sym ? FT / kRefTilesPerWG : 0, tl.list,
                       tl.count, tl.ctrl);
  }
  return hipGetLastError();
}

hipError_t launch_clear_flags(unsigned char* flags, int64_t n, hipStream_t st) {
  const int64_t vec = (n + 15) / 16;
  hipLaunchKernelGGL(clear_kernel, dim3((unsigned)((vec + 255) / 256)), dim3(256), 0, st,
                     reinterpret_cast<uint4*>(flags), vec, (int*)nullptr);
  return hipGetLastError();
}

hipError_t launch_middle(const int* order, int64_t n, int* mid, hipStream_t st) {
  const int groups = (int)((n + 2 * kTile - 1) / (2 * kTile));
  hipLaunchKernelGGL(middle_kernel, dim3((unsigned)((groups + 255) / 256)), dim3(256), 0, st, order,
                     n, groups, mid);
  return hipGetLastError();
}

hipError_t launch_band_list(int ref_tiles, int fit_tiles, int ft, int width, const TileList& tl,
                            hipStream_t st) {
  hipLaunchKernelGGL(band_list_kernel, dim3((unsigned)(fit_tiles / ft)), dim3(64), 0, st,
                     ref_tiles / kRefTilesPerWG, fit_tiles / ft, ft / kRefTilesPerWG, width,
                     tl.list, tl.count);
  return hipGetLastError();
}

hipError_t launch_place_band_list(const unsigned* keys, int dist_bits, const int* order, int64_t n,
                                  int ref_tiles, int fit_tiles, int width, int most,
                                  const TileList& tl, hipStream_t st) {
  if (n < 1 || width < 1 || fit_tiles % kFilterFitTiles) return hipErrorInvalidValue;
  hipLaunchKernelGGL(place_band_list_kernel, dim3((unsigned)(fit_tiles / kFilterFitTiles)), dim3(128),
                     0, st, keys, dist_bits, order, n, ref_tiles / kRefTilesPerWG, width, most,
                     tl.list, tl.count);
  return hipGetLastError();
}

hipError_t launch_places(const int* order, int64_t n, int* place, hipStream_t st) {
  hipLaunchKernelGGL(places_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, order, n,
                     place);
  return hipGetLastError();
}

hipError_t launch_fill_near(unsigned long long* near, int64_t n, hipStream_t st) {
  hipLaunchKernelGGL(fill_near_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, near, n);
  return hipGetLastError();
}

hipError_t launch_near_keys(const unsigned long long* near, int64_t n, int phases, unsigned* keys,
                            int* rows, hipStream_t st) {
  hipLaunchKernelGGL(near_keys_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, near, n,
                     phases, keys, rows);
  return hipGetLastError();
}

hipError_t launch_rank_sort(const unsigned* keys, int* order, int64_t n, hipStream_t st) {
  if (n < 1 || n > kRankSortMax) return hipErrorInvalidValue;
  hipLaunchKernelGGL(rank_sort_kernel, dim3((unsigned)((n + 63) / 64)), dim3(256), 0, st, keys,
                     (int)n, order);
  return hipGetLastError();
}

size_t sort_order_scratch(int64_t n) {
  return (size_t)n * (sizeof(unsigned) + sizeof(int)) + kSortBlocks * 256 * sizeof(int);
}

hipError_t launch_sort_order(const int* leaders, int* rank, int ncells, unsigned* keys,
                             unsigned* keys_out, const int* rows, int* order, int64_t n, void* temp,
                             size_t temp_bytes, hipStream_t st) {
  if (leaders) {
    if (ncells < 1) return hipErrorInvalidValue;
    hipLaunchKernelGGL(cell_rank_kernel, dim3((unsigned)((ncells + 255) / 256)), dim3(256), 0, st,
                       leaders, ncells, rank);
    hipLaunchKernelGGL(rank_keys_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, rank,
                       ncells, n, keys);
  }
  if (n < 1 || n > INT_MAX || temp_bytes < sort_order_scratch(n)) return hipErrorInvalidValue;
  // four rounds, or a multiple that makes no more than kSortBlocks workgroups:
  // each reads the counts of all
  const int rounds = 4 * (int)((n + 1024 * kSortBlocks - 1) / (1024 * kSortBlocks));
  const dim3 grid((unsigned)((n + 256 * rounds - 1) / (256 * rounds)));
  unsigned* const tkeys = (unsigned*)temp;
  int* const trows = (int*)(tkeys + n);
  int* const counts = trows + n;
  for (int pass = 0; pass < 4; ++pass) {
    const unsigned* const kin = pass == 0 ? keys : pass & 1 ? tkeys : keys_out;
    const int* const rin = pass == 0 ? rows : pass & 1 ? trows : order;
    hipLaunchKernelGGL(sort_count_kernel, grid, dim3(256), 0, st, kin, (int)n, rounds, 8 * pass,
                       counts);
    hipLaunchKernelGGL(sort_scatter_kernel, grid, dim3(256), 0, st, kin, rin, (int)n, rounds,
                       8 * pass, counts, pass & 1 ? keys_out : tkeys, pass & 1 ? order : trows);
  }
  return hipGetLastError();
}

}  // namespace mdsctk
