// Structure factor of a detector by interpolation over the detector surface,
// for gfx950 (MI355X).
//
// The direct sum F(q) = sum_j f_j(|q|) w_j exp(-2 pi i q.r_j) of a molecule of
// radius R varies over the detector no faster than the phase of its outermost
// atom: along one detector axis by theta = 2 pi R |dq/du| radians per unit of
// u in [-1, 1], some tens of radians over hundreds of pixels on an oversampled
// detector. So F is summed directly at n_x x n_y nodes, n a little above
// theta, and every pixel interpolates from them:
//
//  1. Surface. q(x, y) is replaced by the polynomial qs(u, v) through 16 x 16
//     of its pixels (Chebyshev form, FP64). What the list has beyond it,
//     d = q - qs, is the FP32 rounding of the list, resolved along the surface's
//     tangents and a fixed normal n, d = alpha dqs/du + beta dqs/dv + gamma n.
//     It must be small, 2 pi R |d| <= 2e-4 at every pixel, otherwise the list is
//     not taken.
//  2. Nodes. u_i = asin(a cos t_i) / asin(a), t_i = (2 i + 1) pi / (2 n), the
//     Chebyshev points stretched towards even spacing (Kosloff & Tal-Ezer,
//     J. Comput. Phys. 104 (1993) 457), with a = 1 / cosh(40 / n): the stretch
//     itself errs by e^-40 times what exp(i theta u) grows by off the axis. (With
//     e^-20.7 atoms all at the molecule's ends, 240 to 330 rad per unit of u, lost
//     4e-7 and 8e-7 of |F|; now 5e-8, with as many nodes.) Beyond theta, the largest
//     phase per unit of t, the Chebyshev coefficients of the phases fall off like Bessel
//     functions, and those of a form factor's e^{-b s^2} like a Gaussian's:
//     n = theta + sqrt((3 theta^(1/3) + 8.5)^2 + 64 b (ds/dt)^2)
//     leaves at most 5e-9 of the steepest phase (rms over u, FP64, up to 560 rad per
//     unit of u; 1e-13 in the median) and 2e-8 of a Gaussian with exponents up to 60.
//  3. Node sums. F and its derivative N = n.dF/dq at the nodes, of large molecules
//     by cells (below), by the arithmetic
//     of the direct kernels (FP64 phase reduced to turns, FP32 sine and
//     cosine, FP32 sums over 64 atoms folded into FP64). On a square detector
//     centred on the beam the nodes come in octants, as its pixels do in the
//     octant kernel (sf_kernels.hip).
//  4. Interpolation along the rows, then along the columns: two small dense
//     products with FP64 weights for F (FP32 for N and for the derivatives of F,
//     whose weights are the derivatives of F's), then per pixel
//     F(q) = e^{-2 pi i q.r0} (F + alpha dF/du + beta dF/dv + gamma N)(u, v),
//     which takes the list's rounding into account to first order (second
//     order: (2 pi R |d|)^2 / 2 <= 2e-8).
//
// The cost is n_x n_y natoms terms instead of npix natoms: 30 times fewer on
// 100,000 atoms x 1024^2 at 0.15 nm (n = 192). The interpolation weights add
// no error of their own: the sum of their squares is 1 over an axis (2 at its ends).
#include "surface.hpp"

#include <algorithm>
#include <cmath>
#include <vector>

#include "form_factor.hpp"
#include "ranges.hpp"

namespace spsim {

namespace {

constexpr int kT = 256;
constexpr int D = kSurfDeg;
constexpr int kLines = kSurfLines;
constexpr double kPi = 3.14159265358979323846;
constexpr float kStretch = 40.0f;       // of the node map, see step 2 above
constexpr double kMaxPhaseDev = 2e-4;   // largest 2 pi R |q - surface|
constexpr double kMaxSpreadDev = 3e-7;  // the same times the spectrum's largest |s_k / sc - 1|
constexpr float kMinWeakest = 0.02f;    // see species_terms
// v_cos_f32 and v_sin_f32 round towards zero: |e^{-i phi}| is short by 3.22e-8 on
// average over the phases (2^26 random ones against FP64), coherently where the
// atoms scatter in phase, so the form factors make up for it.
constexpr double kTrigBias = 3.22e-8;
constexpr float kMaxGauss = 60.0f;      // largest exponent B s^2 over the detector

// a-th of the kSurfDeg sample pixels of an axis: the pixel nearest to the
// Chebyshev-Lobatto point (distinct for 64 pixels and more).
__device__ __forceinline__ int sample_pixel(int a, int n) {
  return (int)rint(0.5 * (1.0 - cospi((double)a / (D - 1))) * (n - 1));
}
__device__ __forceinline__ double pixel_u(int x, int n) { return (2.0 * x - (n - 1)) / (double)(n - 1); }

// Largest (sum for SUM) of N values over the workgroup, given to every thread.
template <int N, bool SUM = false, class T = double>
__device__ __forceinline__ void block_reduce(T (&v)[N]) {
  __shared__ T part[kT / 64][N];
#pragma unroll
  for (int i = 0; i < N; ++i)
    for (int o = 32; o > 0; o >>= 1) {
      const T w = __shfl_xor(v[i], o);
      v[i] = SUM ? v[i] + w : (v[i] < w ? w : v[i]);
    }
  __syncthreads();
  if ((threadIdx.x & 63) == 0)
    for (int i = 0; i < N; ++i) part[threadIdx.x / 64][i] = v[i];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < N; ++i) {
    v[i] = part[0][i];
    for (int w = 1; w < kT / 64; ++w) v[i] = SUM ? v[i] + part[w][i] : (v[i] < part[w][i] ? part[w][i] : v[i]);
  }
}

// ---- 1. scan: the list's surface and deviations, the molecule's radius -------

// C[m][a]: weight of sample a in Chebyshev coefficient m of the polynomial
// through the samples at us: the polynomial at the 16 Chebyshev points
// (barycentric formula), then their cosine transform. cosines[k] = cos(pi k / 32).
__device__ void sample_to_chebyshev(const double *us, const double *cosines, double (*C)[D], double (*tmp)[D]) {
  const int t = threadIdx.x, p = t / D, a = t % D;
  double w = 1.0;
#pragma unroll
  for (int c = 0; c < D; ++c)
    if (c != a) w *= 2.0 * (us[a] - us[c]);
  const double up = cosines[2 * p + 1], d = up - us[a];
  const double v = d == 0.0 ? 0.0 : 1.0 / (w * d);
  tmp[p][a] = v;
  __syncthreads();
  double den = 0.0;
  int hit = -1;
#pragma unroll
  for (int c = 0; c < D; ++c) {
    den += tmp[p][c];
    if (up == us[c]) hit = c;
  }
  __syncthreads();
  tmp[p][a] = hit >= 0 ? (hit == a ? 1.0 : 0.0) : v / den;
  __syncthreads();
  double s = 0.0;
#pragma unroll
  for (int k = 0; k < D; ++k) {
    int j = p * (2 * k + 1) % (4 * D);  // cos(pi j / 32)
    if (j > 2 * D) j = 4 * D - j;
    s += tmp[k][a] * cosines[j];
  }
  C[p][a] = s * (p == 0 ? 1.0 : 2.0) / D;
  __syncthreads();
}

// Chebyshev series of 3 components at u (c[m][3]).
__device__ __forceinline__ void clenshaw3(const double (*c)[3], double u, double out[3]) {
  double b1[3] = {0, 0, 0}, b2[3] = {0, 0, 0};
  const double u2 = 2.0 * u;
#pragma unroll 5
  for (int m = D - 1; m >= 1; --m) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const double b = __builtin_fma(u2, b1[k], c[m][k] - b2[k]);
      b2[k] = b1[k];
      b1[k] = b;
    }
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) out[k] = __builtin_fma(u, b1[k], c[0][k] - b2[k]);
}

// Coefficients along u of the surface's line v: row[m][k] = sum_n T_n(v) coef[n][m][k].
// Threads 0..47.
__device__ __forceinline__ void surface_row(const double (*coef)[D][3], double v, double (*row)[3]) {
  if (threadIdx.x < 3 * D) {
    const int m = threadIdx.x / 3, k = threadIdx.x % 3;
    double t0 = 1.0, t1 = v, s = coef[0][m][k];
    for (int n = 1; n < D; ++n) {
      s = __builtin_fma(t1, coef[n][m][k], s);
      const double t2 = __builtin_fma(2.0 * v, t1, -t0);
      t0 = t1;
      t1 = t2;
    }
    row[m][k] = s;
  }
}

// The same of dq/dv: sum_n n U_{n-1}(v) coef[n][m][k]. Threads 64..111.
__device__ __forceinline__ void surface_row_dv(const double (*coef)[D][3], double v, float (*row)[3]) {
  const int t = (int)threadIdx.x - 64;
  if (t >= 0 && t < 3 * D) {
    const int m = t / 3, k = t % 3;
    double u0 = 0.0, u1 = 1.0, s = 0.0;
    for (int n = 1; n < D; ++n) {
      s = __builtin_fma(n * u1, coef[n][m][k], s);
      const double u2 = __builtin_fma(2.0 * v, u1, -u0);
      u0 = u1;
      u1 = u2;
    }
    row[m][k] = (float)s;
  }
}

// The tangents at u of a line (coefficients c of q, cv of dq/dv), in FP32.
__device__ __forceinline__ void tangents(const double (*c)[3], const float (*cv)[3], float u, float qu[3],
                                         float qv[3]) {
  float a1[3] = {0, 0, 0}, a2[3] = {0, 0, 0}, b1[3] = {0, 0, 0}, b2[3] = {0, 0, 0};
  const float u2 = 2.0f * u;
#pragma unroll 3
  for (int m = D - 1; m >= 1; --m) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const float a = __builtin_fmaf(u2, a1[k], (float)m * (float)c[m][k] - a2[k]);  // sum m c_m U_{m-1}
      a2[k] = a1[k];
      a1[k] = a;
      const float b = __builtin_fmaf(u2, b1[k], cv[m][k] - b2[k]);
      b2[k] = b1[k];
      b1[k] = b;
    }
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    qu[k] = a1[k];
    qv[k] = __builtin_fmaf(u, b1[k], cv[0][k] - b2[k]);
  }
}

__device__ __forceinline__ void cross(const float a[3], const float b[3], float c[3]) {
  c[0] = a[1] * b[2] - a[2] * b[1];
  c[1] = a[2] * b[0] - a[0] * b[2];
  c[2] = a[0] * b[1] - a[1] * b[0];
}
__device__ __forceinline__ float dot(const float a[3], const float b[3]) { return a[0] * b[0] + a[1] * b[1] + a[2] * b[2]; }

// Makes the surface of a detector centred on the beam exactly symmetric: q_x
// odd in u and even in v, q_y even and odd, q_z even in both; and, on a square
// one, q_x(u, v) = q_y(v, u). Coefficients that break it by their rounding
// alone are dropped (what they stood for moves to the deviations). Returns 2,
// 1 (no transposed symmetry) or 0 (none). The normal is that of the middle.
__device__ int symmetrise(double (*Q)[D][3], bool square, float normal[3]) {
  const int n = threadIdx.x / D, m = threadIdx.x % D;  // T_n(v) T_m(u)
  const double x = Q[n][m][0], y = Q[n][m][1], z = Q[n][m][2];
  const bool om = m & 1, on = n & 1;
  // dq/du and dq/dv at u = v = 0 (T_n(0) = cos(n pi / 2), U_{m-1}(0) = sin(m pi / 2)),
  // the coefficients that mirrors and the transposition forbid, all coefficients
  const double au = om && !on ? ((m / 2 + n / 2) & 1 ? -m : m) : 0.0;
  const double av = on && !om ? ((m / 2 + n / 2) & 1 ? -n : n) : 0.0;
  float v[9] = {(float)(au * x),
                (float)(au * y),
                (float)(au * z),
                (float)(av * x),
                (float)(av * y),
                (float)(av * z),
                (float)((om && !on ? 0.0 : fabs(x)) + (on && !om ? 0.0 : fabs(y)) + (om || on ? fabs(z) : 0.0)),
                (float)(fabs(x - Q[m][n][1]) + fabs(z - Q[m][n][2])),
                (float)(fabs(x) + fabs(y) + fabs(z))};
  block_reduce<9, true>(v);
  const int sym = v[6] <= 1e-6f * v[8] ? (square && v[7] <= 1e-6f * v[8] ? 2 : 1) : 0;
  const double xt = Q[m][n][1], yt = Q[m][n][0], zt = Q[m][n][2];
  __syncthreads();
  if (sym > 0) {
    Q[n][m][0] = om && !on ? (sym == 2 ? 0.5 * (x + xt) : x) : 0.0;
    Q[n][m][1] = on && !om ? (sym == 2 ? 0.5 * (y + yt) : y) : 0.0;
    Q[n][m][2] = om || on ? 0.0 : (sym == 2 ? 0.5 * (z + zt) : z);
  }
  __syncthreads();
  cross(v, v + 3, normal);
  if (sym > 0) normal[0] = normal[1] = 0.0f;
  const float len = sqrtf(dot(normal, normal));
  for (int k = 0; k < 3; ++k) normal[k] /= len;
  return sym;
}

struct ScanArgs {
  const float *hkl;
  int nx, ny;
  int list_blocks;  // the last two measure the slopes
  const spsim_hip_atom *atoms;
  const float *atom_b;
  const MolInfo *mols;  // null: the one molecule
  MolInfo one;
  bool centre;  // false: the molecules' centres are the origin
  SurfFit *fit;
  float *dev;
  SurfRecord *records;  // [list_blocks + nmol * kSurfAtomBlocks]
  double *centres;      // [nmol][3]
};

__device__ void scan_list(const ScanArgs &a) {
  __shared__ double C[2][D][D], tmp[D][D], Q[D][D][3], P[D][D][3], row[D][3], us[2][D], cosines[2 * D + 1];
  __shared__ int px[2][D];
  __shared__ float row_v[D][3];
  const int t = threadIdx.x, b = t / D, i = t % D;
  if (t < 2 * D) {
    const int n = b ? a.ny : a.nx;
    px[b][i] = sample_pixel(i, n);
    us[b][i] = pixel_u(px[b][i], n);
  }
  if (t >= 64 && t <= 64 + 2 * D) cosines[t - 64] = cospi((t - 64) / (2.0 * D));
  __syncthreads();
  {
    const size_t p = (size_t)px[1][b] * a.nx + px[0][i];
    for (int k = 0; k < 3; ++k) Q[b][i][k] = a.hkl[3 * p + k];
  }
  // s^2 of the sample pixels, corners among them
  double s2[1] = {(Q[b][i][0] * Q[b][i][0] + Q[b][i][1] * Q[b][i][1] + Q[b][i][2] * Q[b][i][2]) * 2.5e-21};
  if ((int)blockIdx.x == a.list_blocks - 2) block_reduce(s2);
  sample_to_chebyshev(us[0], cosines, C[0], tmp);
  sample_to_chebyshev(us[1], cosines, C[1], tmp);
  // along x: P[b][m], then along y in place of Q
  for (int k = 0; k < 3; ++k) {
    double s = 0.0;
#pragma unroll
    for (int c = 0; c < D; ++c) s = __builtin_fma(C[0][i][c], Q[b][c][k], s);
    P[b][i][k] = s;
  }
  __syncthreads();
  for (int k = 0; k < 3; ++k) {
    double s = 0.0;
#pragma unroll
    for (int c = 0; c < D; ++c) s = __builtin_fma(C[1][b][c], P[c][i][k], s);
    Q[b][i][k] = s;
  }
  __syncthreads();
  float normal[3];
  const int sym = symmetrise(Q, a.nx == a.ny, normal);
  const int rows = a.list_blocks - 2;  // workgroups that take the list's rows
  if ((int)blockIdx.x >= rows) {
    // slopes along one axis on the kLines x kLines Lobatto points: T_m and
    // m U_{m-1} at the points, then dq/du of every row of coefficients, then the points'
    const bool along_y = (int)blockIdx.x == rows + 1;
    __shared__ double T[D][kLines], U[D][kLines], R[D][kLines][3];
    __shared__ unsigned smax[4][kLines];
    if (t < kLines) {
      const double u = cospi((double)t / (kLines - 1));
      double t0 = 1.0, t1 = u, u0 = 0.0, u1 = 1.0;
      for (int m = 0; m < D; ++m) {
        T[m][t] = t0;
        U[m][t] = m * u0;
        const double tn = 2.0 * u * t1 - t0, un = 2.0 * u * u1 - u0;
        t0 = t1;
        t1 = tn;
        u0 = u1;
        u1 = un;
      }
      for (int k = 0; k < 4; ++k) smax[k][t] = 0u;
    }
    __syncthreads();
    for (int c = t; c < D * kLines; c += kT) {
      const int n = c / kLines, j = c % kLines;
      double r[3] = {0, 0, 0};
#pragma unroll
      for (int m = 0; m < D; ++m)
        for (int k = 0; k < 3; ++k) r[k] = __builtin_fma(U[m][j], along_y ? Q[m][n][k] : Q[n][m][k], r[k]);
      for (int k = 0; k < 3; ++k) R[n][j][k] = r[k];
    }
    __syncthreads();
    for (int c = t; c < kLines * kLines; c += kT) {
      const int across = c / kLines, line = c % kLines;
      double d[3] = {0, 0, 0};
#pragma unroll
      for (int n = 0; n < D; ++n)
        for (int k = 0; k < 3; ++k) d[k] = __builtin_fma(T[n][across], R[n][line][k], d[k]);
      // non-negative floats order as their bits
      atomicMax(&smax[3][line], __float_as_uint((float)sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2])));
      for (int k = 0; k < 3; ++k) atomicMax(&smax[k][line], __float_as_uint((float)fabs(d[k])));
    }
    __syncthreads();
    if (t < kLines) {
      SurfSlopes &out = along_y ? a.fit->slope_y : a.fit->slope_x;
      out.all[t] = __uint_as_float(smax[3][t]);
      for (int k = 0; k < 3; ++k) out.part[k][t] = __uint_as_float(smax[k][t]);
    }
    if (t == 0) a.records[blockIdx.x] = SurfRecord{0.0, 0.0, 0.0f, 0.0f, 0, 0};
    if (!along_y) {
      if (t == 0) {
        a.fit->s2max = (float)s2[0];
        a.fit->sym = sym;
        for (int k = 0; k < 3; ++k) a.fit->normal[k] = normal[k];
      }
      for (int c = t; c < D * D * 3; c += kT) (&a.fit->coef[0][0][0])[c] = (&Q[0][0][0])[c];
    }
    return;
  }
  double m[2] = {0, 0};
  for (int y = blockIdx.x; y < a.ny; y += rows) {
    __syncthreads();
    surface_row(Q, pixel_u(y, a.ny), row);
    surface_row_dv(Q, pixel_u(y, a.ny), row_v);
    __syncthreads();
    for (int x = t; x < a.nx; x += kT) {
      double s[3];
      float qu[3], qv[3], d[3], uv[3], vn[3], nu[3];
      const double u = pixel_u(x, a.nx);
      clenshaw3(row, u, s);
      tangents(row, row_v, (float)u, qu, qv);
      const size_t p = 3 * ((size_t)y * a.nx + x);
#pragma unroll
      for (int k = 0; k < 3; ++k) d[k] = (float)((double)a.hkl[p + k] - s[k]);
      cross(qu, qv, uv);
      cross(qv, normal, vn);
      cross(normal, qu, nu);
      const float inv = 1.0f / dot(qu, vn);
      const float al = dot(d, vn) * inv, be = dot(d, nu) * inv, ga = dot(d, uv) * inv;
      a.dev[p] = al;
      a.dev[p + 1] = be;
      a.dev[p + 2] = ga;
      const float size = fabsf(al) * sqrtf(dot(qu, qu)) + fabsf(be) * sqrtf(dot(qv, qv)) + fabsf(ga);
      if (!(size < 1e30f)) m[1] = 1.0;
      m[0] = fmax(m[0], (double)size);
    }
  }
  block_reduce(m);
  if (t == 0) a.records[blockIdx.x] = SurfRecord{m[0], 0.0, 0.0f, 0.0f, m[1] > 0.0, 0};
}

// The molecule's centre is the mean of 1024 evenly spaced atoms: any point near
// the middle serves, and every workgroup forms the same one.
__device__ void scan_atoms(const ScanArgs &a) {
  const int t = threadIdx.x;
  const int mol = ((int)blockIdx.x - a.list_blocks) / kSurfAtomBlocks;
  const int part = ((int)blockIdx.x - a.list_blocks) % kSurfAtomBlocks;
  const MolInfo mi = a.mols ? a.mols[mol] : a.one;
  const int begin = mi.atom_begin, n = mi.atom_end - begin;
  const spsim_hip_atom *atoms = a.atoms + begin;
  double c[3] = {0, 0, 0};
  if (n > 0 && a.centre)
    for (int i = 0; i < 4; ++i) {
      const spsim_hip_atom at = atoms[(int)((long long)(4 * t + i) * n / (4 * kT))];
      c[0] += at.x;
      c[1] += at.y;
      c[2] += at.z;
    }
  block_reduce<3, true>(c);
  for (int k = 0; k < 3; ++k) c[k] /= 4.0 * kT;
  if (part == 0 && t == 0)
    for (int k = 0; k < 3; ++k) a.centres[3 * mol + k] = c[k];
  // |r - r0|^2, -B, B, not finite
  double m[4] = {0.0, -3.4e38, -3.4e38, fabs(c[0]) + fabs(c[1]) + fabs(c[2]) < 1e30 ? 0.0 : 1.0};
  for (long long j = part * kT + t; j < n; j += kSurfAtomBlocks * kT) {
    const spsim_hip_atom at = atoms[j];
    const double x = at.x - c[0], y = at.y - c[1], z = at.z - c[2];
    const double d2 = x * x + y * y + z * z;
    if (!(d2 < 1e30) || !(fabsf(at.w) < 3.4e38f)) m[3] = 1.0;
    m[0] = fmax(m[0], d2);
    if (a.atom_b) {
      const float b = a.atom_b[begin + j];
      if (!(fabsf(b) < 1e30f)) m[3] = 1.0;
      m[1] = fmax(m[1], -(double)b);
      m[2] = fmax(m[2], (double)b);
    }
  }
  block_reduce(m);
  if (t == 0)
    a.records[blockIdx.x] = SurfRecord{0.0, m[0], (float)-m[1], (float)m[2], m[3] > 0.0, 0};
}

__global__ __launch_bounds__(kT, 3) void surface_scan_kernel(ScanArgs a) {
  if ((int)blockIdx.x < a.list_blocks)
    scan_list(a);
  else
    scan_atoms(a);
}

// ---- 2. nodes -------------------------------------------------------------------

// The stretch parameter of n nodes, and the nodes that atoms within `radius` and
// within a box of half edges h need at that stretch. 2 % are added to the slopes
// for their sampling.
__host__ __device__ inline float axis_stretch(int n) { return 1.0f / coshf(kStretch / n); }

// On the line u = cos(pi k / (kLines - 1)), x = u asin(a): s = sin(x) / a,
// |du/dt| = sqrt(1 - s^2) a / (asin(a) cos(x)), here times asin(a). Lines mirrored
// about the middle share them.
__host__ __device__ inline float line_density(int k, float a, float as) {
#ifdef __HIP_DEVICE_COMPILE__
  const float x = fabsf(__builtin_amdgcn_cosf(0.5f * k / (kLines - 1))) * as;
  const float sx = __builtin_amdgcn_sinf(x * (float)(0.5 / kPi)), cx = __builtin_amdgcn_cosf(x * (float)(0.5 / kPi));
  return __builtin_amdgcn_sqrtf(fmaxf(0.0f, a * a - sx * sx)) * __builtin_amdgcn_rcpf(fmaxf(cx, 1e-6f));
#else
  const float x = std::fabs(std::cos((float)kPi * k / (kLines - 1))) * as;
  const float sx = std::sin(x), cx = std::cos(x);
  return std::sqrt(std::max(0.0f, a * a - sx * sx)) / std::max(cx, 1e-6f);
#endif
}

// density(k) as line_density at the stretch whose asin is as; steepest(): the largest
// slope.all[k] density(k), asked for behind the densities; b: the largest Gaussian
// coefficient of the terms, A^2.
template <class Density, class Steepest>
__host__ __device__ inline float axis_need(const SurfSlopes &slope, float radius, const float *h, float b, float as,
                                           Density density, Steepest steepest) {
  float w = 0.0f;
  for (int k = 0; k < kLines; ++k) {
    const float box = slope.part[0][k] * h[0] + slope.part[1][k] * h[1] + slope.part[2][k] * h[2];
    w = fmaxf(w, fminf(slope.all[k] * radius, box) * density(k));
  }
  const float theta = 1.02f * 2.0f * (float)kPi * w / as;
  const float tail = 3.0f * cbrtf(theta) + 8.5f, s = 0.5e-10f * steepest() / as;  // ds per node angle
  return theta + sqrtf(tail * tail + 64.0f * fmaxf(b, 0.0f) * s * s);
}

__device__ __forceinline__ float axis_need(const SurfSlopes &slope, float radius, const float *h, float b, float a) {
  const float as = asinf(a);
  float steepest = 0.0f;
  return axis_need(
      slope, radius, h, b, as,
      [&](int k) {
        const float d = line_density(k, a, as);
        steepest = fmaxf(steepest, slope.all[k] * d);
        return d;
      },
      [&] { return steepest; });
}

enum class SurfKind { kSum, kSpectrum, kAdjoint };

__host__ __device__ inline bool worth(double nodes_x, double nodes_y, double nx, double ny, double natoms,
                                      SurfKind kind) {
  // Issue cycles per lane: a term of the node sums 60 (140 with a spectrum, 100
  // in the adjoint), of the direct sums 26 to 45 (130, 109); the interpolation
  // 25 per node row and pixel. Measured on the MI355X.
  const double node = kind == SurfKind::kSum ? 60.0 : (kind == SurfKind::kSpectrum ? 140.0 : 100.0);
  const double direct = kind == SurfKind::kSum ? 26.0 : (kind == SurfKind::kSpectrum ? 130.0 : 109.0);
  const double surf = nodes_x * nodes_y * natoms * node + 25.0 * (nx * ny * nodes_y + nx * nodes_x * nodes_y);
  return surf < 0.8 * direct * nx * ny * natoms;
}

__host__ __device__ inline bool smooth(const SurfMol &m, float s2max) {
  return !m.bad && 2.0 * kPi * m.radius * m.dev <= kMaxPhaseDev && m.weakest >= kMinWeakest &&
         m.b_smooth * s2max <= kMaxGauss;
}

// Amplitude of a term over the detector, per species: the interpolation's error
// is relative to the strongest part of the pattern, the direct sum's to the
// pixel's own terms, so terms that fade below kMinWeakest of their value at
// the beam are left to the direct sum.
__host__ __device__ inline void species_terms(const float *c, float Bs, float bmin, float bmax, float s2max,
                                              float *b_smooth, float *weakest) {
  float f0 = c[8], f1 = c[8], b = 0.0f;
  for (int i = 0; i < 4; ++i) {
    f0 += c[i];
    f1 += c[i] * expf(-c[4 + i] * s2max);
    b = fmaxf(b, fabsf(c[4 + i]));
  }
  const float lo = Bs + bmin, hi = Bs + bmax;
  const float e0 = fmaxf(1.0f, expf(-lo * s2max)), e1 = fminf(1.0f, expf(-hi * s2max));
  const float ratio = fabsf(f1) * e1 / (fabsf(f0) * e0);
  *b_smooth = fmaxf(*b_smooth, b + fmaxf(fabsf(lo), fabsf(hi)));
  *weakest = ratio < *weakest || !(ratio < 1e30f) ? (ratio < 1e30f ? ratio : 0.0f) : *weakest;
}

// Atom records of the node sums: position relative to the centre, rotated
// (FP64), the amplitude w and its product with n.r; with per-atom B, log2 of the
// amplitude, n.r and B.
struct __align__(16) NodeAtom {
  double x, y, z;
  float w, n, b, pad;
};
static_assert(sizeof(NodeAtom) == 48, "node-sum atom record");

// Cell index along an axis of g cells over [-extent, extent].
__device__ __forceinline__ int cell_index(double x, double extent, int g) {
  return min(g - 1, max(0, (int)((x / extent + 1.0) * 0.5 * g)));
}

__device__ __forceinline__ void prepare_atoms(const SurfJob &jb, bool has_b, int first, int step) {
  NodeAtom *out = (NodeAtom *)jb.prep;
  const SurfCells &c = jb.c;
  for (long long j = first; j < jb.natoms; j += step) {
    const spsim_hip_atom at = jb.atoms[j];
    const double x = at.x - jb.r0[0], y = at.y - jb.r0[1], z = at.z - jb.r0[2];
    NodeAtom r;
    if (jb.has_rot) {
      const double *R = jb.rot;
      r.x = __builtin_fma(R[6], z, __builtin_fma(R[3], y, R[0] * x));
      r.y = __builtin_fma(R[7], z, __builtin_fma(R[4], y, R[1] * x));
      r.z = __builtin_fma(R[8], z, __builtin_fma(R[5], y, R[2] * x));
    } else {
      r.x = x;
      r.y = y;
      r.z = z;
    }
    const float n = jb.normal[0] * (float)r.x + jb.normal[1] * (float)r.y + jb.normal[2] * (float)r.z;
    r.w = has_b ? log2f(at.w) : at.w;
    r.n = has_b ? n : at.w * n;
    r.b = has_b ? jb.atom_b[j] : 0.0f;
    r.pad = 0.0f;
    out[j] = r;
    if (c.g > 0)
      c.id[j] = (unsigned short)((cell_index(r.z, c.extent, c.gz) * c.g + cell_index(r.y, c.extent, c.g)) * c.g +
                                 cell_index(r.x, c.extent, c.g));
    if (c.g > 0 && j == jb.natoms - 1)  // whole words for the sort
      for (int p = jb.natoms; p < (jb.natoms + 7) / 8 * 8; ++p) c.id[p] = 0xffff;
  }
}

// Octants of an n x n node grid (n even).
__host__ __device__ inline int node_octants(int n) { return n / 2 * (n / 2 + 1) / 2; }

// Nodes per lane of the node sums and tiles of 256 lanes. An octant (8 nodes)
// shares phases between its nodes: 321 issue cycles per atom against 57 per
// node alone; four nodes per lane share an atom's LDS read (one: 75). The tiling
// with the least work; on few terms one node per lane, for the most work items
// (on 1024 nodes x 5,000 atoms, 13 us against 24 us with four).
__host__ __device__ inline void node_tiling(int nx, int ny, bool octants, long long natoms, int *per_lane, int *tiles) {
  const int nodes = nx * ny;
  if (nodes * natoms < 1LL << 25) {
    *per_lane = 1;
    *tiles = (nodes + kT - 1) / kT;
    return;
  }
  const int t2 = (nodes + 2 * kT - 1) / (2 * kT), t4 = (nodes + 4 * kT - 1) / (4 * kT);
  const int t8 = (node_octants(nx) + kT - 1) / kT;
  *per_lane = t4 * 228 <= t2 * 120 ? 4 : 2;
  *tiles = *per_lane == 4 ? t4 : t2;
  if (octants && t8 * 321 < *tiles * (*per_lane == 4 ? 228 : 120)) {
    *per_lane = 8;
    *tiles = t8;
  }
}

// Node e of a lane, of a work item's tile: its index, or -1 where there is none.
// Octant t stands for the node (x, y), x <= y = the row of t in the triangle,
// its mirrors, and the transposed node with its mirrors.
__device__ __forceinline__ void octant_node(int t, int &x, int &y) {
  int yy = (int)((sqrtf(8.0f * (float)t + 1.0f) - 1.0f) * 0.5f);
  while ((yy + 1) * (yy + 2) / 2 <= t) ++yy;
  while (yy * (yy + 1) / 2 > t) --yy;
  y = yy;
  x = t - yy * (yy + 1) / 2;
}
template <int T = kT>  // lanes per tile
__device__ __forceinline__ int node_index(int per_lane, int nxn, int nyn, int tile, int e, int lane) {
  if (per_lane == 8) {
    const int t = tile * T + lane;
    if (t >= node_octants(nyn)) return -1;
    int x, y;
    octant_node(t, x, y);
    if (e >= 4 && x == y) return -1;  // on the diagonal both quads are the same nodes: one writes them
    const int m = nyn - 1;
    const int i = e < 4 ? x : y, k = e < 4 ? y : x;  // mirrored in x for odd e, in y for e & 2
    return ((e & 1) ? m - i : i) * nyn + ((e & 2) ? m - k : k);
  }
  const int node = tile * per_lane * T + e * T + lane;
  return node < nxn * nyn ? node : -1;
}
__device__ __forceinline__ int node_index(const SurfJob &jb, int tile, int e, int lane) {
  return node_index(jb.per_lane, jb.sh.ax.n, jb.sh.ay.n, tile, e, lane);
}

// Time of the node sums in atoms per lane with s atom ranges per tile: rounds
// of `slots` resident workgroups, each of an atom range and a fixed part (the
// form factors and the loop's start, about 40 atoms), and the ranges' partial
// sums, which cost about half an atom each.
__host__ __device__ inline float splits_cost(int s, int tiles, int natoms, int slots) {
  const int rounds = (tiles * s + slots - 1) / slots;
  return rounds * ((float)natoms / s + 40.0f) + (s > 1 ? 0.5f * s + 40.0f : 0.0f);
}

struct PlanArgs {
  SurfJob job;  // template: pointers and sizes set, the choice left open
  const SurfFit *fit;
  const SurfRecord *records;
  int list_blocks;
  const double *centres;
  const float *ff;
  float b_global;
  bool has_b;
  int slots;       // resident workgroups of the node sums
  int slot_cap;    // partial slots that fit
  int max_nx, max_ny;  // nodes that fit the workspace
  int max_cells;       // 0: no sums by cells
  long long max_cell_sums, max_cell_rows;
  SurfKind kind;
  double scale, spread;  // of a spectrum: largest s_k, largest |s_k / sc - 1|
  SurfJob *out;
  // adjoint: pixel values 2 g F e^{2 pi i q.r0} from the list, F and g
  const float *hkl;
  const float2 *F;
  const float *gI;
  float2 *pixels;
};

__device__ __forceinline__ void prepare_pixels(const PlanArgs &a, const SurfJob &jb, int first, int step) {
  for (int p = first; p < jb.nx * jb.ny; p += step) {
    const double t = __builtin_fma((double)a.hkl[3 * p + 2], jb.r0[2],
                                   __builtin_fma((double)a.hkl[3 * p + 1], jb.r0[1], (double)a.hkl[3 * p] * jb.r0[0]));
    double sn, cs;
    sincospi(2.0 * __builtin_amdgcn_fract(t), &sn, &cs);
    const float2 f = a.F[p];
    const double g = 2.0 * (double)a.gI[p];
    a.pixels[p] = make_float2((float)(g * (f.x * cs - f.y * sn)), (float)(g * (f.x * sn + f.y * cs)));
  }
}

// Interpolation weights of one axis, and in FP32 with their derivatives in u
// (DERIV; node-major [n][npix]), one wave per pixel x at u: barycentric formula in s = cos t, whose
// weights at the Chebyshev points are (-1)^i sin t_i. With r_i = w_i / (s - s_i):
// l_i = r_i / sum r, dl_i/ds = l_i (sum r_j / (s - s_j) / sum r - 1 / (s - s_i)).
template <bool DERIV = true>
__device__ __forceinline__ void weight_column(const SurfAxis &ax, double u, int x, int npix, const double *sn,
                                              const double *wn, double *__restrict__ out, float2 *__restrict__ out32) {
  const int lane = threadIdx.x & 63;
  double sx, cx;
  sincospi(u * (ax.asin_a / kPi), &sx, &cx);
  const double s = sx / ax.a, ds = ax.asin_a * cx / ax.a;
  double sum = 0.0, sum2 = 0.0;
  int hit = -1;
  for (int i = lane; i < ax.n; i += 64) {
    const double d = s - sn[i];
    if (fabs(d) < 1e-13) {
      hit = i;
    } else {
      const double r = wn[i] / d;
      sum += r;
      sum2 += r / d;
    }
  }
  for (int o = 32; o > 0; o >>= 1) {
    sum += __shfl_xor(sum, o);
    sum2 += __shfl_xor(sum2, o);
    hit = max(hit, __shfl_xor(hit, o));
  }
  // on a node h: l is its unit vector, dl_i/ds = w_i / w_h / (s_h - s_i), and
  // minus their sum at h itself
  for (int i = lane; i < ax.n; i += 64) {
    const double d = s - sn[i], r = wn[i] / d;
    const size_t o = (size_t)i * npix + x;
    if (hit >= 0) {
      out[o] = i == hit ? 1.0 : 0.0;
      if constexpr (DERIV)
        out32[o] = make_float2(i == hit ? 1.0f : 0.0f, (float)(ds * (i == hit ? -sum / wn[hit] : r / wn[hit])));
    } else {
      const double l = r / sum;
      out[o] = l;
      if constexpr (DERIV)
        out32[o] = make_float2((float)l, (float)(ds * l * (sum2 / sum - 1.0 / d)));
    }
  }
}

__device__ __forceinline__ double node_u(const SurfAxis &ax, int i) {
  return asin(ax.a * cospi((2 * i + 1) / (2.0 * ax.n))) / ax.asin_a;
}

// LDS arrays of build().
struct BuildLds {
  double snx[kSurfMaxNodes], wnx[kSurfMaxNodes], sny[kSurfMaxNodes], wny[kSurfMaxNodes];
  double coef[D][D][3], row[D][3];
};

// Barycentric nodes and weights of an axis.
__device__ __forceinline__ void axis_tables(const SurfAxis &ax, double *sn, double *wn) {
  for (int i = threadIdx.x; i < ax.n; i += kT) {
    const double ph = (2 * i + 1) / (2.0 * ax.n);
    sn[i] = cospi(ph);
    wn[i] = (i & 1) ? -sinpi(ph) : sinpi(ph);
  }
}

// q at the nodes ax x ay, node (i, k) -> index i ay.n + k: a row of 16 nodes is
// contiguous for the first product.
__device__ void build_nodes(const SurfFit *fit, const SurfAxis &ax, const SurfAxis &ay, double *out, BuildLds &l) {
  const int t = threadIdx.x;
  for (int i = t; i < D * D * 3; i += kT) (&l.coef[0][0][0])[i] = (&fit->coef[0][0][0])[i];
  for (int i = t; i < ax.n; i += kT) l.snx[i] = node_u(ax, i);
  for (int i = t; i < ay.n; i += kT) l.sny[i] = node_u(ay, i);
  for (int k = blockIdx.x; k < ay.n; k += gridDim.x) {
    __syncthreads();
    surface_row(l.coef, l.sny[k], l.row);
    __syncthreads();
    for (int i = t; i < ax.n; i += kT) {
      double q[3];
      clenshaw3(l.row, l.snx[i], q);
      double *o = out + 3 * ((size_t)i * ay.n + k);
      o[0] = q[0];
      o[1] = q[1];
      o[2] = q[2];
    }
  }
}

// Part 0: the weights of both axes, part 1: the node q of a shape, spread over
// gridDim.x workgroups. Called by every thread.
__device__ void build(int part, const SurfFit *fit, const SurfShape &sh, int nx, int ny, BuildLds &l) {
  if (part == 1) build_nodes(fit, sh.ax, sh.ay, sh.nodes, l);
  if (part != 0) return;
  axis_tables(sh.ax, l.snx, l.wnx);
  axis_tables(sh.ay, l.sny, l.wny);
  __syncthreads();
  const int waves = kT / 64, wave = threadIdx.x / 64;
  for (int r = (int)blockIdx.x * waves + wave; r < nx + ny; r += (int)gridDim.x * waves) {
    if (r < nx)
      weight_column(sh.ax, pixel_u(r, nx), r, nx, l.snx, l.wnx, sh.tx, sh.tx32);
    else
      weight_column(sh.ay, pixel_u(r - nx, ny), r - nx, ny, l.sny, l.wny, sh.ty, sh.ty32);
  }
}

// The same for the coarse nodes of a molecule's cells, onto the pattern's nodes.
__device__ void build_coarse(int part, const SurfFit *fit, const SurfCoarse &co, BuildLds &l) {
  if (part == 1) build_nodes(fit, co.ax, co.ay, co.nodes, l);
  if (part != 0) return;
  axis_tables(co.ax, l.snx, l.wnx);
  axis_tables(co.ay, l.sny, l.wny);
  __syncthreads();
  const int waves = kT / 64, wave = threadIdx.x / 64, nx = co.fx.n, ny = co.fy.n;
  for (int r = (int)blockIdx.x * waves + wave; r < nx + ny; r += (int)gridDim.x * waves) {
    if (r < nx)
      weight_column<false>(co.ax, node_u(co.fx, r), r, nx, l.snx, l.wnx, co.wx, nullptr);
    else
      weight_column<false>(co.ay, node_u(co.fy, r - nx), r - nx, ny, l.sny, l.wny, co.wy, nullptr);
  }
}

// Box grids that are tried: cells across the beam and along it.
constexpr int kCellGrids = 4, kMaxCells = 512;
// Most atoms per work item of a cell's sums: at most 512 ranges besides one
// of every cell.
__host__ __device__ inline int cell_range(int natoms) { return 256 * (natoms / (256 * 512) + 1); }
__host__ __device__ inline void cell_grid(int k, int *g, int *gz) {
  *g = k == 0 ? 4 : (k == 1 ? 6 : 8);
  *gz = k == 0 ? 2 : (k == 1 ? 3 : (k == 2 ? 4 : 8));
}
constexpr int kCellMinNodes = 16, kCellMaxNodes = 128;  // of a cell's sums, per axis

// The same for the nodes of a cell, in tiles of 64 lanes.
__host__ __device__ inline void cell_tiling(int nx, int ny, bool octants, int *per_lane, int *tiles) {
  const int nodes = nx * ny, t2 = (nodes + 127) / 128, t4 = (nodes + 255) / 256, t8 = (node_octants(nx) + 63) / 64;
  *per_lane = t4 * 228 <= t2 * 120 ? 4 : 2;
  *tiles = *per_lane == 4 ? t4 : t2;
  if (octants && t8 * 321 < *tiles * (*per_lane == 4 ? 228 : 120)) {
    *per_lane = 8;
    *tiles = t8;
  }
}

// Issue cycles over all lanes of a pattern's node sums (nx x ny nodes), and of
// the same by cells with mx x my nodes each: the sums, the two products
// (290 cycles per 16 x 16 x 4 block, an FP64 sine and cosine per node and cell)
// and the products' memory (about 33 cycles a byte). The weights of the sums and
// the products order the grids of boxes as they measured: on 100,000 atoms and 192^2
// nodes 108 cells of 64^2 nodes take 239 us, 256 of 52^2 260 us (0.6 for the
// products had them the other way round).
__host__ __device__ inline double sums_cost(int nx, int ny, bool octants, double natoms, int *per_lane, int *tiles) {
  node_tiling(nx, ny, octants, 1LL << 25, per_lane, tiles);
  return (double)*tiles * kT * (*per_lane == 8 ? 321.0 : 57.0 * *per_lane) * natoms;
}
__host__ __device__ inline double cells_cost(int nx, int ny, int mx, int my, int ncells, bool octants, double natoms) {
  int per_lane, tiles;
  cell_tiling(mx, my, octants, &per_lane, &tiles);
  const double sums = tiles * 64.0 * (per_lane == 8 ? 321.0 : 57.0 * per_lane) * natoms;
  auto up = [](int n) { return (n + 15) / 16; };
  const double rows = 290.0 * up(nx) * up(my) * (mx / 4), cols = up(nx) * up(ny) * (290.0 * (my / 4) + 2000.0);
  return 1.2 * sums + 0.8 * ncells * (64.0 * (rows + cols) + 33.0 * 48.0 * my * nx);
}

// What the scan found about a molecule on its list, in *out (thread 0).
__device__ void fold_records(const SurfRecord *list, int nlist, const SurfRecord *atoms, const spsim_hip_segment *segs,
                             int nsegs, const float *ff, float b_global, bool has_b, float s2max, SurfMol *out) {
  const int t = threadIdx.x;
  double m[5] = {0, 0, -3.4e38, -3.4e38, 0};  // dev, r2, -B, B, not finite
  for (int i = t; i < nlist + kSurfAtomBlocks; i += kT) {
    const SurfRecord r = i < nlist ? list[i] : atoms[i - nlist];
    m[0] = fmax(m[0], r.dev);
    m[1] = fmax(m[1], r.r2);
    if (i >= nlist) {
      m[2] = fmax(m[2], -(double)r.bmin);
      m[3] = fmax(m[3], (double)r.bmax);
    }
    if (r.bad) m[4] = 1.0;
  }
  block_reduce(m);
  // every form-factor row that is used, one thread each
  float bs = 0.0f, weak = 1.0f;
  double e[3] = {0.0, 0.0, 0.0};  // Gaussian, -weakest, no order for cells
  for (int i = t; i < nsegs; i += kT) {
    if (segs[i].count < 0 || (i > 0 && segs[i].start < segs[i - 1].start + segs[i - 1].count)) e[2] = 1.0;
    if (segs[i].count <= 0) continue;  // no atom of it: the sums never look at its species
    const int sp = segs[i].species;
    species_terms(ff + sp * SPSIM_HIP_FF_STRIDE, sp == SPSIM_HIP_UNIT_SPECIES ? 0.0f : b_global,
                  has_b ? (float)-m[2] : 0.0f, has_b ? (float)m[3] : 0.0f, s2max, &bs, &weak);
  }
  e[0] = bs;
  e[1] = -(double)weak;
  if (nsegs > SPSIM_HIP_NSPECIES) e[2] = 1.0;  // more than surface_sort_kernel counts
  block_reduce(e);
  if (t == 0) *out = SurfMol{sqrt(m[1]), m[0], (float)e[0], (float)-e[1], m[4] > 0.0, e[2] == 0.0};
}

// One workgroup per molecule.
struct DigestArgs {
  const SurfFit *fit;
  const SurfRecord *records;
  int list_blocks;
  const MolInfo *mols;
  MolInfo one;
  const spsim_hip_segment *segs;
  const float *ff;
  float b_global;
  bool has_b;
  const double *centres;
  SurfHead *head;
  SurfDigest *out;
};

__global__ __launch_bounds__(kT) void surface_digest_kernel(DigestArgs a) {
  const int m = blockIdx.x, t = threadIdx.x;
  const MolInfo mi = a.mols ? a.mols[m] : a.one;
  SurfDigest d;
  fold_records(a.records, a.list_blocks, a.records + a.list_blocks + (size_t)m * kSurfAtomBlocks, a.segs + mi.seg_begin,
               mi.nseg, a.ff, a.b_global, a.has_b, a.fit->s2max, &d.mol);
  if (t == 0) {
    for (int k = 0; k < 3; ++k) d.centre[k] = a.centres[3 * m + k];
    a.out[m] = d;
  }
  if (m > 0) return;
  for (int i = t; i < (int)(sizeof(SurfSlopes) / sizeof(float)); i += kT) {
    ((float *)&a.head->slope_x)[i] = ((const float *)&a.fit->slope_x)[i];
    ((float *)&a.head->slope_y)[i] = ((const float *)&a.fit->slope_y)[i];
  }
  if (t == 0) {
    a.head->s2max = a.fit->s2max;
    for (int k = 0; k < 3; ++k) a.head->normal[k] = a.fit->normal[k];
    a.head->sym = a.fit->sym;
  }
}

// Partial sums over the cells, for about 1024 workgroups of the second product.
__host__ __device__ inline int cell_splits(int nx, int ny, int count, long long slot_cap) {
  const int wgs = ((nx + 31) / 32) * ((ny + 31) / 32) * count;
  int s = 1024 / wgs;
  const long long nodes = ((long long)nx * ny + kT - 1) / kT * kT;
  s = s < 1 ? 1 : (s > 32 ? 32 : s);
  while (s > 1 && nodes * s > slot_cap) --s;
  return s;
}

// *out = *in by the workgroup (one lane would take a struct through scratch).
template <class T>
__device__ __forceinline__ void copy_words(T *out, const T *in) {
  static_assert(sizeof(T) % 4 == 0, "whole words");
  for (int i = threadIdx.x; i < (int)(sizeof(T) / 4); i += kT) ((unsigned *)out)[i] = ((const unsigned *)in)[i];
}

// The grid of boxes that costs least, or -1 when the plain sums do. max_*: what
// the workspace holds.
__device__ int choose_cells(const PlanArgs &a, int nx, int ny, bool octants, const int (*n)[2]) {
  __shared__ float cost[kCellGrids + 1];
  const int k = threadIdx.x;
  int per_lane, tiles;
  if (k < kCellGrids) {  // one grid per lane
    int g, gz;
    cell_grid(k, &g, &gz);
    const int mx = n[k][0], my = n[k][1], ncells = g * g * gz;
    const bool fits = mx <= kCellMaxNodes && my <= kCellMaxNodes && ncells <= a.max_cells &&
                      (long long)(a.job.natoms / cell_range(a.job.natoms) + ncells) * mx * my <= a.max_cell_sums &&
                      (long long)ncells * my * nx <= a.max_cell_rows;
    cost[k] = fits ? (float)cells_cost(nx, ny, mx, my, ncells, octants && mx == my, a.job.natoms) : 3e38f;
  } else if (k == kCellGrids) {
    cost[k] = (float)(0.7 * sums_cost(nx, ny, octants, a.job.natoms, &per_lane, &tiles) - 4e9);
  }
  __syncthreads();
  int best = kCellGrids;
  for (int i = 0; i < kCellGrids; ++i) best = cost[i] < cost[best] ? i : best;
  return best < kCellGrids ? best : -1;
}

__global__ __launch_bounds__(kT) void surface_plan_kernel(PlanArgs a) {
  __shared__ BuildLds lds;
  __shared__ SurfMol mol;
  __shared__ int best[2], split[1], cell_best[kCellGrids][2];
  __shared__ SurfJob job;
  const int t = threadIdx.x;
  fold_records(a.records, a.list_blocks, a.records + a.list_blocks, a.job.segs, a.job.nsegs, a.ff, a.b_global, a.has_b,
               a.fit->s2max, &mol);
  if (t == 0) {
    mol.radius *= a.scale;
    best[0] = best[1] = 1 << 30;
    for (int k = 0; k < kCellGrids; ++k) cell_best[k][0] = cell_best[k][1] = 1 << 30;
  }
  __syncthreads();
  {  // smallest sufficient node count of each axis, one candidate per thread
    const int axis = t / 128, n = kSurfMinNodes + 4 * (t % 128);
    const SurfSlopes &slope = axis ? a.fit->slope_y : a.fit->slope_x;
    const float r = (float)mol.radius, h[3] = {r, r, r};
    if (n <= kSurfMaxNodes && axis_need(slope, r, h, mol.b_smooth, axis_stretch(n)) <= (float)n)
      atomicMin(&best[axis], n);
  }
  if (a.max_cells > 0)  // and of the cells of every grid of boxes
    for (int i = t; i < kCellGrids * 2 * 32; i += kT) {
      const int k = i / 64, axis = i / 32 % 2, n = kCellMinNodes + 4 * (i % 32);
      int g, gz;
      cell_grid(k, &g, &gz);
      const SurfSlopes &slope = axis ? a.fit->slope_y : a.fit->slope_x;
      const float r = (float)mol.radius, h[3] = {r / g, r / g, r / gz};
      if (n <= kCellMaxNodes && axis_need(slope, sqrtf(h[0] * h[0] + h[1] * h[1] + h[2] * h[2]), h,
                                          mol.b_smooth, axis_stretch(n)) <= (float)n)
        atomicMin(&cell_best[k][axis], n);
    }
  __syncthreads();
  const int nx = best[0], ny = best[1];
  // N is taken at the spectrum's centre scale, so it is off by the spread
  const bool ok = smooth(mol, a.fit->s2max) && 2.0 * kPi * mol.radius * mol.dev * a.spread <= kMaxSpreadDev &&
                  nx <= a.max_nx && ny <= a.max_ny &&
                  worth(nx, ny, a.job.nx, a.job.ny, a.job.natoms, a.kind);
  if (!ok) {
    if (blockIdx.x == 0 && blockIdx.y == 0 && t == 0) a.out->ok = 0;
    return;
  }
  int per_lane, tiles, grid = -1;
  const bool octants = a.fit->sym == 2 && nx == ny && a.kind == SurfKind::kSum;
  if (a.max_cells > 0 && mol.ordered) grid = choose_cells(a, nx, ny, octants, cell_best);
  node_tiling(nx, ny, octants, a.job.natoms, &per_lane, &tiles);
  copy_words(&job, &a.job);
  __syncthreads();
  if (grid >= 0) {  // F and N come as partial sums over cells, node by node
    per_lane = 1;
    tiles = (nx * ny + kT - 1) / kT;
  }
  const int tile = per_lane * kT;
  if (t < 64) {  // the cheapest number of atom ranges, two candidates per lane
    float c = 3.0e38f;
    int n = 1;
    for (int s = t + 1; s <= kSurfMaxSplits; s += 64)
      if (s == 1 || ((long long)tiles * tile * s <= a.slot_cap && a.job.natoms / s >= 32)) {
        const float k = splits_cost(s, tiles, a.job.natoms, a.slots);
        if (k < c) {
          c = k;
          n = s;
        }
      }
    for (int o = 32; o > 0; o >>= 1) {
      const float c2 = __shfl_xor(c, o);
      const int n2 = __shfl_xor(n, o);
      if (c2 < c || (c2 == c && n2 < n)) {
        c = c2;
        n = n2;
      }
    }
    if (t == 0) split[0] = grid >= 0 ? cell_splits(nx, ny, 1, a.slot_cap) : n;
  } else if (t == 64) {
    job.ok = 1;
    job.sh.ax = SurfAxis{nx, axis_stretch(nx), 0.0};
    job.sh.ay = SurfAxis{ny, axis_stretch(ny), 0.0};
    job.sh.ax.asin_a = asin(job.sh.ax.a);
    job.sh.ay.asin_a = asin(job.sh.ay.a);
    job.per_lane = per_lane;
    job.tiles = tiles;
    job.c.g = 0;
    if (grid >= 0) {
      SurfCells &c = job.c;
      cell_grid(grid, &c.g, &c.gz);
      c.extent = mol.radius;
      c.co.ax = SurfAxis{cell_best[grid][0], axis_stretch(cell_best[grid][0]), 0.0};
      c.co.ay = SurfAxis{cell_best[grid][1], axis_stretch(cell_best[grid][1]), 0.0};
      c.co.ax.asin_a = asin(c.co.ax.a);
      c.co.ay.asin_a = asin(c.co.ay.a);
      c.co.fx = job.sh.ax;
      c.co.fy = job.sh.ay;
      cell_tiling(c.co.ax.n, c.co.ay.n, octants && c.co.ax.n == c.co.ay.n, &c.per_lane, &c.tiles);
    }
    for (int k = 0; k < 3; ++k) {
      job.r0[k] = a.centres[k];
      job.normal[k] = a.fit->normal[k];
    }
  }
  __syncthreads();
  if (t == 0) job.splits = split[0];
  __syncthreads();
  if (blockIdx.x == 0 && blockIdx.y == 0) copy_words(a.out, &job);
  build(blockIdx.y, a.fit, job.sh, job.nx, job.ny, lds);
  if (job.c.g > 0) build_coarse((int)blockIdx.y - 3, a.fit, job.c.co, lds);
  if (blockIdx.y == 2) {
    const int first = (int)(blockIdx.x * kT) + t, step = (int)gridDim.x * kT;
    if (a.kind == SurfKind::kAdjoint)
      prepare_pixels(a, job, first, step);
    else
      prepare_atoms(job, a.has_b, first, step);
  }
}

__global__ __launch_bounds__(kT) void surface_tables_kernel(const SurfFit *fit, const SurfShape *shapes, int nx, int ny) {
  __shared__ BuildLds lds;
  build(blockIdx.y, fit, shapes[blockIdx.z], nx, ny, lds);
}

__global__ __launch_bounds__(kT) void surface_coarse_kernel(const SurfFit *fit, const SurfCoarse *coarse) {
  __shared__ BuildLds lds;
  build_coarse(blockIdx.y, fit, coarse[blockIdx.z], lds);
}

// ---- 3. node sums ---------------------------------------------------------------
//
// One work item: a tile of nodes (node_tiling) x one atom range, whose records
// are staged in LDS 256 at a time; every lane reads the same record, and its
// terms share the read. Per node and atom: 3 FP64 FMAs, a fraction and a
// conversion, a sine and cosine, 4 FP32 FMAs (F and N): 57 issue cycles; an
// octant's 8 nodes share 9 FP64 operations, 5 fractions, conversions, sines and
// cosines: 40 per node (100,000 atoms with B, 188^2 nodes: 1.14 ms, two nodes
// per lane 1.9 ms with three gradient sums instead of N). (The records through scalar loads instead, one node per
// lane: 128 cycles; the waves drift apart and miss the scalar cache.) A tile's
// atom ranges leave partial sums, which surface_reduce_kernel adds in range
// order (added by the tile's last workgroup instead, 64 ranges took 30 us: one
// lane per node waits for every slot). The form factor is evaluated in FP64:
// its rounding at a node would be shared by all the pixels around it.

constexpr int kNodeChunk = 256;  // atoms staged at once
constexpr int kNodeFold = 64;  // atoms per FP32 partial sum

__device__ __forceinline__ double form_factor64(const float *__restrict__ c, double s2, float B) {
  double f = c[8] * exp(-(double)B * s2);
#pragma unroll
  for (int i = 0; i < 4; ++i) f += c[i] * exp(-((double)c[4 + i] + B) * s2);
  return f;
}

// The spectrum travels in the kernel's arguments only where there is one.
struct NoSpectrum {};
template <bool SPEC>
struct SpectrumArg {
  using type = NoSpectrum;
};
template <>
struct SpectrumArg<true> {
  using type = Spectrum;
};

// One term of a spectrum: U(t) = sum_k W_k e^{-2 pi i s_k t} as (ur, -ui) for
// the FP64 phase t = q.r in turns, by the polynomials within their range, else
// by the sample sum with each s_k t reduced to turns in FP64, as in spectrum_sum
// (sf_kernels.hip).
__device__ __forceinline__ void spectrum_term(const Spectrum &sp, int ns, double t, float &ur, float &ui) {
  const double tc = sp.sc * t;
  const float tf = (float)tc;
  if (__builtin_fabsf(tf) <= sp.tlim) {
    asm volatile("");  // keeps the polynomials under the branch, not formed for every atom
    const float ph = (float)__builtin_amdgcn_fract(tc);
    const float cs = __builtin_amdgcn_cosf(ph);
    const float sn = __builtin_amdgcn_sinf(ph);
    const float v = tf * sp.inv_tlim;
    const float u = v * v;
    float gc = sp.p[kSpectrumDegree], gq = sp.q[kSpectrumDegree];
#pragma unroll
    for (int d = kSpectrumDegree - 1; d >= 0; --d) {
      gc = __builtin_fmaf(gc, u, sp.p[d]);
      gq = __builtin_fmaf(gq, u, sp.q[d]);
    }
    const float gs = v * gq;
    ur = __builtin_fmaf(cs, gc, -sn * gs);
    ui = __builtin_fmaf(sn, gc, cs * gs);
    return;
  }
  float sr = 0.0f, si = 0.0f;
  int m = 0;
  do {  // at least one sample
    const float ph = (float)__builtin_amdgcn_fract(sp.s[m] * t);
    sr = __builtin_fmaf(sp.w[m], __builtin_amdgcn_cosf(ph), sr);
    si = __builtin_fmaf(sp.w[m], __builtin_amdgcn_sinf(ph), si);
  } while (++m < ns);
  ur = sr;
  ui = si;
}

// A lane's sums of node e: a partial sum, or F and N = -2 pi i sum w f n.r e^{-i phi}.
__device__ __forceinline__ void store_node(const SurfJob &jb, int tile, int split, int e, double fc, double fs, float nc,
                                           float ns) {
  if (jb.splits > 1) {
    const size_t o = ((size_t)tile * jb.splits + split) * jb.per_lane * kT + e * kT + threadIdx.x;
    jb.slot_f[o] = make_double2(fc, fs);
    jb.slot_n[o] = make_float2(nc, ns);
    return;
  }
  const int node = node_index(jb, tile, e, threadIdx.x);
  if (node < 0) return;
  jb.f[node] = make_double2(fc, -fs);
  jb.n[node] = make_float2(-2.0f * (float)kPi * ns, -2.0f * (float)kPi * nc);
}

// The nodes of a grid and the atoms [a_begin, a_end) of a work item.
struct NodeWork {
  const double *nodes;
  int nxn, nyn, per_lane;
  const NodeAtom *atoms;
  const spsim_hip_segment *segs;
  int nsegs, a_begin, a_end;
};

// Lanes of a wave see the LDS writes of the others.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Runs body(first, count) over the LDS chunks of a work item's atoms, at most
// kNodeFold atoms at a time; form(species) is called once per species. WAVE: the
// item is one wave's, with an sm of its own for 64 atoms.
template <bool WAVE, class Form, class Body>
__device__ __forceinline__ void over_atoms(const NodeWork &jb, NodeAtom *sm, Form form, Body body) {
  for (int sg = 0; sg < jb.nsegs; ++sg) {
    const spsim_hip_segment seg = jb.segs[sg];
    const int lo = max(seg.start, jb.a_begin), hi = min(seg.start + seg.count, jb.a_end);
    if (lo >= hi) continue;
    form(seg.species);
    constexpr int kChunk = WAVE ? 64 : kNodeChunk;
    const int t = WAVE ? threadIdx.x & 63 : threadIdx.x;
    for (int c0 = lo; c0 < hi; c0 += kChunk) {
      const int n = min(kChunk, hi - c0);
      WAVE ? wave_sync() : __syncthreads();
      if (t < n) sm[t] = jb.atoms[c0 + t];
      WAVE ? wave_sync() : __syncthreads();
      for (int j0 = 0; j0 < n; j0 += kNodeFold) body(j0, min(n, j0 + kNodeFold));
    }
  }
}

// K nodes per lane. SPEC: a wavelength spectrum, the sample sum in place of the
// sine and cosine (spectrum_term), and N at the centre scale.
template <int K, bool HAS_B, bool SPEC, bool WAVE, class Store>
__device__ __forceinline__ void node_item(const NodeWork &jb, int tile, const float *__restrict__ ff, float b_global,
                                          const typename SpectrumArg<SPEC>::type &sp, NodeAtom *sm, Store store) {
  constexpr int kUnroll = K == 1 ? 4 : (K == 2 ? 2 : 1);
  const int lane = WAVE ? threadIdx.x & 63 : threadIdx.x;
  double qx[K], qy[K], qz[K], s2[K], f[K], Fc[K], Fs[K];
  float nl2[K], Nc[K], Ns[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const double *q = jb.nodes + 3 * (size_t)max(0, node_index<WAVE ? 64 : kT>(K, jb.nxn, jb.nyn, tile, k, lane));
    qx[k] = q[0];
    qy[k] = q[1];
    qz[k] = q[2];
    s2[k] = (qx[k] * qx[k] + qy[k] * qy[k] + qz[k] * qz[k]) * 2.5e-21;
    nl2[k] = (float)(-s2[k] * kLog2e);
    f[k] = Fc[k] = Fs[k] = 0.0;
    Nc[k] = Ns[k] = 0.0f;
  }
  over_atoms<WAVE>(
      jb, sm,
      [&](int species) {
#pragma unroll
        for (int k = 0; k < K; ++k)
          f[k] = (1.0 + kTrigBias) * form_factor64(ff + species * SPSIM_HIP_FF_STRIDE, s2[k],
                                                   species == SPSIM_HIP_UNIT_SPECIES ? 0.0f : b_global);
      },
      [&](int j0, int j1) {
        float c[K][2], s[K][2];
#pragma unroll
        for (int k = 0; k < K; ++k) c[k][0] = c[k][1] = s[k][0] = s[k][1] = 0.0f;
#pragma unroll kUnroll
        for (int j = j0; j < j1; ++j) {
          const NodeAtom at = sm[j];
#pragma unroll
          for (int k = 0; k < K; ++k) {
            const double t = __builtin_fma(qz[k], at.z, __builtin_fma(qy[k], at.y, qx[k] * at.x));
            float cs, sn;
            if constexpr (SPEC) {
              spectrum_term(sp, sp.n, t, cs, sn);
            } else {
              const float ph = (float)__builtin_amdgcn_fract(t);
              cs = __builtin_amdgcn_cosf(ph);
              sn = __builtin_amdgcn_sinf(ph);
            }
            if constexpr (HAS_B) {
              const float w = __builtin_amdgcn_exp2f(__builtin_fmaf(at.b, nl2[k], at.w));
              cs *= w;
              sn *= w;
              c[k][0] += cs;
              s[k][0] += sn;
            } else {
              c[k][0] = __builtin_fmaf(at.w, cs, c[k][0]);
              s[k][0] = __builtin_fmaf(at.w, sn, s[k][0]);
            }
            c[k][1] = __builtin_fmaf(at.n, cs, c[k][1]);
            s[k][1] = __builtin_fmaf(at.n, sn, s[k][1]);
          }
        }
#pragma unroll
        for (int k = 0; k < K; ++k) {
          Fc[k] = __builtin_fma(f[k], (double)c[k][0], Fc[k]);
          Fs[k] = __builtin_fma(f[k], (double)s[k][0], Fs[k]);
          Nc[k] = __builtin_fmaf((float)f[k], c[k][1], Nc[k]);
          Ns[k] = __builtin_fmaf((float)f[k], s[k][1], Ns[k]);
        }
      });
#pragma unroll
  for (int k = 0; k < K; ++k) {
    float scale = 1.0f;
    if constexpr (SPEC) scale = (float)sp.sc;
    store(k, Fc[k], Fs[k], scale * Nc[k], scale * Ns[k]);
  }
}

// One octant per lane: the phases a + b, a - b of the node (x, y) and of its
// transposed node with a = q_x r_x, b = q_y r_y, c = q_z r_z, and from their sines and
// cosines the four real sums P, Q per angle, as in octant_sum (sf_kernels.hip),
// once weighted by w e^{-2 pi i c} (F) and once by n.r times that (N).
template <bool HAS_B, bool WAVE, class Store>
__device__ __forceinline__ void octant_item(const NodeWork &jb, int tile, const float *__restrict__ ff, float b_global,
                                            NodeAtom *sm, Store store) {
  const int lane = WAVE ? threadIdx.x & 63 : threadIdx.x;
  const double *q = jb.nodes + 3 * (size_t)max(0, node_index<WAVE ? 64 : kT>(8, jb.nxn, jb.nyn, tile, 0, lane));
  const double qx = q[0], qy = q[1], qz = q[2];
  const double s2 = (qx * qx + qy * qy + qz * qz) * 2.5e-21;
  const float nl2 = (float)(-s2 * kLog2e);
  double f = 0.0, Fc[8], Fs[8];
  float Nc[8], Ns[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    Fc[i] = Fs[i] = 0.0;
    Nc[i] = Ns[i] = 0.0f;
  }
  over_atoms<WAVE>(
      jb, sm,
      [&](int species) {
        f = (1.0 + 2.0 * kTrigBias) * form_factor64(ff + species * SPSIM_HIP_FF_STRIDE, s2,
                                                    species == SPSIM_HIP_UNIT_SPECIES ? 0.0f : b_global);
      },
      [&](int j0, int j1) {
        // [half][F, N][P, Q over a + b, P, Q over a - b][by cos c, by sin c]
        float S[2][2][4][2];
#pragma unroll
        for (int i = 0; i < 32; ++i) (&S[0][0][0][0])[i] = 0.0f;
        for (int j = j0; j < j1; ++j) {
          const NodeAtom at = sm[j];
          const double tc = qz * at.z;
          const double ta[2] = {qx * at.x, qy * at.x}, tb[2] = {qy * at.y, qx * at.y};
          const float fc = (float)__builtin_amdgcn_fract(tc);
          float u[2][2];  // [F, N][cos c, sin c]
          u[0][0] = __builtin_amdgcn_cosf(fc);
          u[0][1] = __builtin_amdgcn_sinf(fc);
          if constexpr (HAS_B) {
            const float w = __builtin_amdgcn_exp2f(__builtin_fmaf(at.b, nl2, at.w));
            u[0][0] *= w;
            u[0][1] *= w;
            u[1][0] = at.n * u[0][0];
            u[1][1] = at.n * u[0][1];
          } else {
            u[1][0] = at.n * u[0][0];
            u[1][1] = at.n * u[0][1];
            u[0][0] *= at.w;
            u[0][1] *= at.w;
          }
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const float fs = (float)__builtin_amdgcn_fract(ta[h] + tb[h]);
            const float fd = (float)__builtin_amdgcn_fract(ta[h] - tb[h]);
            const float v[4] = {__builtin_amdgcn_cosf(fs), __builtin_amdgcn_sinf(fs), __builtin_amdgcn_cosf(fd),
                                __builtin_amdgcn_sinf(fd)};
#pragma unroll
            for (int w = 0; w < 2; ++w)
#pragma unroll
              for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int k = 0; k < 2; ++k) S[h][w][i][k] = __builtin_fmaf(u[w][k], v[i], S[h][w][i][k]);
          }
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            // c + (a + b), c - (a - b), c + (a - b), c - (a + b): cosine sums P cos c
            // -/+ Q sin c, sine sums P sin c +/- Q cos c
            const int i = e == 0 || e == 3 ? 0 : 2;
            const bool minus = e == 1 || e == 3;  // the angle enters with a minus
            const float(*F)[2] = S[h][0], (*N)[2] = S[h][1];
            const double pf = F[i][0], ps = F[i][1], qf = F[i + 1][0], qs = F[i + 1][1];
            Fc[4 * h + e] = __builtin_fma(f, minus ? pf + qs : pf - qs, Fc[4 * h + e]);
            Fs[4 * h + e] = __builtin_fma(f, minus ? ps - qf : ps + qf, Fs[4 * h + e]);
            const float f32 = (float)f;
            Nc[4 * h + e] = __builtin_fmaf(f32, minus ? N[i][0] + N[i + 1][1] : N[i][0] - N[i + 1][1], Nc[4 * h + e]);
            Ns[4 * h + e] = __builtin_fmaf(f32, minus ? N[i][1] - N[i + 1][0] : N[i][1] + N[i + 1][0], Ns[4 * h + e]);
          }
        }
      });
#pragma unroll
  for (int e = 0; e < 8; ++e) store(e, Fc[e], Fs[e], Nc[e], Ns[e]);
}

template <bool HAS_B, bool SPEC, bool WAVE, class Store>
__device__ __forceinline__ void any_item(const NodeWork &w, int tile, const float *__restrict__ ff, float b_global,
                                         const typename SpectrumArg<SPEC>::type &sp, NodeAtom *sm, Store store) {
  if constexpr (!SPEC) {
    if (w.per_lane == 8) {
      octant_item<HAS_B, WAVE>(w, tile, ff, b_global, sm, store);
      return;
    }
  }
  if (w.per_lane == 4)
    node_item<4, HAS_B, SPEC, WAVE>(w, tile, ff, b_global, sp, sm, store);
  else if (w.per_lane == 2)
    node_item<2, HAS_B, SPEC, WAVE>(w, tile, ff, b_global, sp, sm, store);
  else
    node_item<1, HAS_B, SPEC, WAVE>(w, tile, ff, b_global, sp, sm, store);
}

template <bool HAS_B, bool SPEC>
__global__ __launch_bounds__(kT) void surface_nodes_kernel(const SurfJob *jobs, const SurfItem *items, int nitems,
                                                           const float *__restrict__ ff, float b_global,
                                                           typename SpectrumArg<SPEC>::type sp) {
  __shared__ NodeAtom sm[kNodeChunk];
  if (!items) {  // one pattern: every (tile, range) of job 0
    if (!jobs->ok || jobs->c.g > 0) return;
    nitems = jobs->tiles * jobs->splits;
  }
  for (int it = blockIdx.x; it < nitems; it += gridDim.x) {
    const SurfItem m = items ? items[it] : SurfItem{0, it % jobs->tiles, it / jobs->tiles, 0};
    const SurfJob &jb = jobs[m.job];
    const NodeWork w{jb.sh.nodes,
                     jb.sh.ax.n,
                     jb.sh.ay.n,
                     jb.per_lane,
                     (const NodeAtom *)jb.prep,
                     jb.segs,
                     jb.nsegs,
                     range_begin(jb.natoms, m.split, jb.splits),
                     range_begin(jb.natoms, m.split + 1, jb.splits)};
    any_item<HAS_B, SPEC, false>(w, m.tile, ff, b_global, sp, sm, [&](int e, double fc, double fs, float nc, float ns) {
      store_node(jb, m.tile, m.split, e, fc, fs, nc, ns);
    });
  }
}

// ---- 3b. node sums by cells -------------------------------------------------------
//
// On many nodes the atoms are summed by cells: g x g x gz boxes, each of whose
// sums about the box's centre varies 1 / g as fast over the detector and
// needs that many fewer nodes per axis; its values there are interpolated to the
// pattern's nodes like the pattern's to the pixels (FP64 products for F, FP32 for
// N), turned by the centre's phase and added up. Terms fall with the square of
// the coarse nodes, the interpolation grows with the cells: cells_cost. On
// 100,000 atoms with B and 192^2 nodes, 108 cells of 64^2 nodes: 27 us for the
// sort, 162 us for the sums, 36 and 86 us for the products, against 1140 us for
// the plain sums (at 188^2).

// The records of one cell (blockIdx.x), in their order, which is that of the
// species: every wave goes over one section of the atoms' cell indexes, 512 at a
// time, counts its atoms in this cell and in lower ones, and lists its own behind
// those of the waves before it; the workgroup then copies the records. The cell's
// ranges are numbered from start / range length + cell, which leaves each room
// enough. Bound by the look at every index in every cell, two to a word (one at a
// time: 52 us instead of 45 us on 8 x 50,000 atoms).
constexpr int kSortT = 1024;

__global__ __launch_bounds__(kSortT) void surface_sort_kernel(const SurfJob *jobs, int first) {
  const SurfJob &jb = jobs[first + blockIdx.z];
  const SurfCells &c = jb.c;
  const int cell = blockIdx.x, t = threadIdx.x, lane = t & 63, wave = t / 64;
  if (!jb.ok || cell >= c.g * c.g * c.gz) return;
  constexpr int kWaves = kSortT / 64;
  __shared__ int counts[kWaves][2], seg_count[SPSIM_HIP_NSPECIES];
  __shared__ spsim_hip_segment seg[SPSIM_HIP_NSPECIES];
  // read once: the stores below might change the job for all the compiler knows
  const unsigned short *ids = c.id;
  int *order = c.order;
  const NodeAtom *in = (const NodeAtom *)jb.prep;
  NodeAtom *out = (NodeAtom *)c.sorted;
  const bool has_b = jb.atom_b != nullptr;
  const int n = jb.natoms, nsegs = jb.nsegs, len = cell_range(n);
  const int section = (n + 512 * kWaves - 1) / (512 * kWaves) * 512, n8 = (n + 7) / 8 * 8;
  const int lo = min(n8, section * wave), hi = min(n8, section * (wave + 1));
  // two indexes to a word, both below 0x8000 or padding: a half's top bit stays
  // set in (w | tops) - c where the half is at least c
  constexpr unsigned kTops = 0x80008000u;
  const unsigned c1 = (unsigned)cell * 0x10001u, c2 = c1 + 0x10001u;
  int lower = 0, upto = 0;  // indexes below this cell, and up to it
#pragma unroll 2
  for (int j = lo + 8 * lane; j < hi; j += 512) {
    const uint4 v = *(const uint4 *)(ids + j);
    auto word = [&](unsigned w) {
      w |= kTops;
      lower += __popc(~(w - c1) & kTops);
      upto += __popc(~(w - c2) & kTops);
    };
    word(v.x);
    word(v.y);
    word(v.z);
    word(v.w);
  }
  int own = upto - lower;
  for (int o = 32; o > 0; o >>= 1) {
    lower += __shfl_xor(lower, o);
    own += __shfl_xor(own, o);
  }
  if (lane == 0) {
    counts[wave][0] = lower;
    counts[wave][1] = own;
  }
  if (t < jb.nsegs) {
    seg_count[t] = 0;
    seg[t] = jb.segs[t];
  }
  __syncthreads();
  int start = 0, total = 0, at = 0;
  for (int i = 0; i < kWaves; ++i) {
    start += counts[i][0];
    at += i < wave ? counts[i][1] : 0;
    total += counts[i][1];
  }
  at += start;
  for (int j = lo; j < hi && own > 0; j += 512) {
    unsigned mask = 0;  // of the 8 indexes from j + 8 lane on, those in this cell
    if (j + 8 * lane < hi) {
      const uint4 v = *(const uint4 *)(ids + j + 8 * lane);
      auto word = [&](unsigned w, int k) {
        const unsigned e = ~(((w ^ c1) | kTops) - 0x10001u) & kTops & ~w;
        mask |= (e >> 15 & 1u | e >> 30) << k;
      };
      word(v.x, 0);
      word(v.y, 2);
      word(v.z, 4);
      word(v.w, 6);
    }
    if (__ballot(mask != 0) == 0) continue;
    int before = __popc(mask);  // of the lanes below: inclusive scan, less its own
    const int mine = before;
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(before, o);
      before += lane >= o ? v : 0;
    }
    int to = at + before - mine;
    at += __shfl(before, 63);
    own -= __shfl(before, 63);
    for (; mask; mask &= mask - 1) order[to++] = j + 8 * lane + __ffs(mask) - 1;
  }
  const int ix[3] = {cell % c.g, cell / c.g % c.g, cell / (c.g * c.g)};
  double centre[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) centre[k] = c.extent * ((2 * ix[k] + 1) / (double)(k < 2 ? c.g : c.gz) - 1.0);
  __threadfence_block();
  __syncthreads();
  for (int i = start + t; i < start + total; i += kSortT) {
    const int a = order[i];
    NodeAtom r = in[a];
    int sg = 0;
    while (sg < nsegs - 1 && a >= seg[sg].start + seg[sg].count) ++sg;
    r.x -= centre[0];
    r.y -= centre[1];
    r.z -= centre[2];
    if (a < seg[sg].start || a >= seg[sg].start + seg[sg].count) {  // of no species: not summed
      r.w = has_b ? -INFINITY : 0.0f;
      r.n = 0.0f;
    }
    out[i] = r;
    atomicAdd(&seg_count[sg], 1);
  }
  __syncthreads();
  if (t == 0) {
    spsim_hip_segment *segs = c.segs + (size_t)cell * jb.nsegs;
    int s = start;
    for (int i = 0; i < jb.nsegs; ++i) {
      segs[i] = spsim_hip_segment{s, seg_count[i], seg[i].species, 0};
      s += seg_count[i];
    }
    SurfCell out_cell;
#pragma unroll
    for (int k = 0; k < 3; ++k) out_cell.centre[k] = centre[k];
    out_cell.start = start;
    out_cell.count = total;
    out_cell.range0 = start / len + cell;
    out_cell.ranges = (total + len - 1) / len;
    c.cells[cell] = out_cell;
  }
  const int r0 = start / len + cell, used = (total + len - 1) / len;
  const int r1 = (start + total) / len + cell + 1;
  for (int r = r0 + t; r < r1; r += kSortT) c.range_cell[r] = r < r0 + used ? cell : -1;
}

// One (range, tile of 64 lanes) per workgroup at a time, of pattern
// first + blockIdx.y: every wave sums a quarter of the range's atoms, and the first
// one adds them up. Bound by the vector units, busy 87 % (77 % of the issue slots;
// ranges of 1024 atoms take 204 us for 161 us, their last ones run alone).
template <bool HAS_B>
__global__ __launch_bounds__(kT, 4) void surface_cell_nodes_kernel(const SurfJob *jobs, int first,
                                                                   const float *__restrict__ ff, float b_global) {
  constexpr int kWaves = kT / 64;
  __shared__ union {
    NodeAtom sm[kWaves][64];
    struct {
      double f[kWaves - 1][2][8][64];
      float n[kWaves - 1][2][8][64];
    } part;
  } lds;
  const SurfJob &jb = jobs[first + blockIdx.y];
  const SurfCells &c = jb.c;
  if (!jb.ok || c.g == 0) return;
  const int len = cell_range(jb.natoms), items = (jb.natoms / len + c.g * c.g * c.gz) * c.tiles;
  for (int it = blockIdx.x; it < items; it += gridDim.x) {
    const int range = it / c.tiles, tile = it % c.tiles, id = c.range_cell[range];
    if (id < 0) continue;
    const SurfCell cell = c.cells[id];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x & 63;
    const int r = range - cell.range0;
    const int begin = cell.start + range_begin(cell.count, r, cell.ranges);
    const int count = cell.start + range_begin(cell.count, r + 1, cell.ranges) - begin;
    const int nxn = c.co.ax.n, nyn = c.co.ay.n;
    const NodeWork w{c.co.nodes,
                     nxn,
                     nyn,
                     c.per_lane,
                     (const NodeAtom *)c.sorted,
                     c.segs + (size_t)id * jb.nsegs,
                     jb.nsegs,
                     begin + range_begin(count, wave, kWaves),
                     begin + range_begin(count, wave + 1, kWaves)};
    NoSpectrum none;
    double fc[8] = {}, fs[8] = {};
    float nc[8] = {}, ns[8] = {};
    any_item<HAS_B, false, true>(w, tile, ff, b_global, none, lds.sm[wave],
                                 [&](int e, double c0, double s0, float c1, float s1) {
                                   fc[e] = c0;
                                   fs[e] = s0;
                                   nc[e] = c1;
                                   ns[e] = s1;
                                 });
    __syncthreads();
    if (wave > 0)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        lds.part.f[wave - 1][0][e][lane] = fc[e];
        lds.part.f[wave - 1][1][e][lane] = fs[e];
        lds.part.n[wave - 1][0][e][lane] = nc[e];
        lds.part.n[wave - 1][1][e][lane] = ns[e];
      }
    __syncthreads();
    double2 *f = c.f + (size_t)range * nxn * nyn;
    float2 *n = c.n + (size_t)range * nxn * nyn;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      if (wave > 0 || e >= c.per_lane) break;
      for (int k = 0; k < kWaves - 1; ++k) {
        fc[e] += lds.part.f[k][0][e][lane];
        fs[e] += lds.part.f[k][1][e][lane];
        nc[e] += lds.part.n[k][0][e][lane];
        ns[e] += lds.part.n[k][1][e][lane];
      }
      const int node = node_index<64>(c.per_lane, nxn, nyn, tile, e, lane);
      if (node < 0) continue;
      f[node] = make_double2(fc[e], -fs[e]);
      n[node] = make_float2(-2.0f * (float)kPi * ns[e], -2.0f * (float)kPi * nc[e]);
    }
    __syncthreads();
  }
}

// Adds the atom ranges of every node: one lane per node for F (blockIdx.y = 0)
// and one for N, 16 ranges in flight.
__global__ __launch_bounds__(kT) void surface_reduce_kernel(const SurfJob *jobs, int first) {
  const SurfJob &jb = jobs[first + blockIdx.z];
  if (!jb.ok || jb.splits == 1) return;
  const int id = (int)blockIdx.x * kT + threadIdx.x, size = jb.per_lane * kT;
  const int tile = id / size, splits = jb.splits;
  if (tile >= jb.tiles) return;
  const int node = node_index(jb, tile, id % size / kT, id % kT);
  if (node < 0) return;
  const size_t at = (size_t)tile * splits * size + id % size;
  if (blockIdx.y == 0) {
    double c = 0.0, s = 0.0;
#pragma unroll 16
    for (int i = 0; i < splits; ++i) {
      const double2 v = jb.slot_f[at + (size_t)i * size];
      c += v.x;
      s += v.y;
    }
    jb.f[node] = make_double2(c, -s);
  } else {
    float c = 0.0f, s = 0.0f;
#pragma unroll 16
    for (int i = 0; i < splits; ++i) {
      const float2 v = jb.slot_n[at + (size_t)i * size];
      c += v.x;
      s += v.y;
    }
    jb.n[node] = make_float2(-2.0f * (float)kPi * s, -2.0f * (float)kPi * c);
  }
}

// ---- 4. interpolation -----------------------------------------------------------
//
// Both products run on the matrix units, in FP64 for F and FP32 for N and
// the derivatives (16 x 16 x 4 products; 105 and 40 cycles each, as fast as the vector FMAs
// they replace: 76 and 42). Lane l of an FP64 product holds rows
// l / 16 + 4 r (r = 0..3) of column l % 16, of an FP32 product rows
// 4 (l / 16) + r: the FP32 products take their rows in the order `prow`, so
// that a lane's F, N and derivatives belong to the same pixels. (Scalar operands and vector
// FMAs instead: 18 us for the rows of a 256 x 256 detector at 28 nodes, where
// each step waits for its scalar loads.)

typedef double double4v __attribute__((ext_vector_type(4)));
typedef float float4v __attribute__((ext_vector_type(4)));

template <int G>
struct Fields {
  double4v re, im;
  float4v g[G];
};

template <int G>
__device__ __forceinline__ void clear(Fields<G> &a) {
  a.re = a.im = double4v{0, 0, 0, 0};
#pragma unroll
  for (int c = 0; c < G; ++c) a.g[c] = float4v{0, 0, 0, 0};
}

__device__ __forceinline__ float4v mfma32(float a, float b, float4v c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ double4v mfma64(double a, double b, double4v c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Row of an FP32 product that puts a lane's results on its FP64 rows.
__device__ __forceinline__ int prow(int m) { return m / 4 + 4 * (m % 4); }

// A cell's sums onto the pattern's node columns: tf[cell][k][x] =
// sum_i f[i][k] wx[i][x]: 16 coarse rows of a cell per workgroup at a time, whose
// sums over the ranges it gathers in LDS first, every wave then for every
// fourth 16 columns; blockIdx.y: pattern. 36 us on 108 cells of 64^2 nodes in
// 490 ranges, bound by their loads. (Read by every wave as it goes, 16 columns
// each: 71 us, a chain of loads and products; 32 columns each: 91 us.)
__global__ __launch_bounds__(kT) void surface_cell_rows_kernel(const SurfJob *jobs, int first) {
  __shared__ double2 sf[kCellMaxNodes * 16];
  __shared__ float2 sn[kCellMaxNodes * 16];
  const SurfJob &jb = jobs[first + blockIdx.y];
  const SurfCells &c = jb.c;
  if (!jb.ok || c.g == 0) return;
  const int mxn = c.co.ax.n, myn = c.co.ay.n, nxn = c.co.fx.n;
  const int wave = threadIdx.x / 64, l = threadIdx.x & 63, m = l & 15, gq = l >> 4;
  const int tiles_k = (myn + 15) / 16, items = tiles_k * c.g * c.g * c.gz;
  const size_t step = (size_t)mxn * myn;
  for (int it = blockIdx.x; it < items; it += gridDim.x) {
    const int id = it / tiles_k, k0 = it % tiles_k * 16;
    const SurfCell cell = c.cells[id];
    if (cell.count == 0) continue;
    // rows and columns past the end repeat the last one and are not stored
    for (int e = threadIdx.x; e < 16 * mxn; e += kT) {
      const size_t node = cell.range0 * step + (size_t)(e / 16) * myn + min(k0 + e % 16, myn - 1);
      double re = 0.0, im = 0.0;
      float nr = 0.0f, ni = 0.0f;
#pragma unroll 4
      for (int r = 0; r < cell.ranges; ++r) {
        const double2 f = c.f[node + r * step];
        const float2 n = c.n[node + r * step];
        re += f.x;
        im += f.y;
        nr += n.x;
        ni += n.y;
      }
      sf[e] = make_double2(re, im);
      sn[e] = make_float2(nr, ni);
    }
    __syncthreads();
    for (int x = wave * 16 + m; x - m < nxn; x += kT / 4) {
      const double *wx = c.co.wx + (size_t)gq * nxn + min(x, nxn - 1);
      Fields<2> acc;
      clear(acc);
#pragma unroll 4
      for (int i = 0; i < mxn; i += 4) {
        const double2 f = sf[16 * (i + gq) + m];
        const float2 n = sn[16 * (i + gq) + prow(m)];
        const double b = wx[(size_t)i * nxn];
        acc.re = mfma64(f.x, b, acc.re);
        acc.im = mfma64(f.y, b, acc.im);
        acc.g[0] = mfma32(n.x, (float)b, acc.g[0]);
        acc.g[1] = mfma32(n.y, (float)b, acc.g[1]);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int k = k0 + gq + 4 * r;
        if (k >= myn || x >= nxn) continue;
        const size_t o = ((size_t)id * myn + k) * nxn + x;
        c.tf[o] = make_double2(acc.re[r], acc.im[r]);
        c.tn[o] = make_float2(acc.g[0][r], acc.g[1][r]);
      }
    }
    __syncthreads();
  }
}

// And onto its rows, F(x, y) = sum_cells e^{-2 pi i q.c} sum_k wy[k][y] tf[cell][k][x] at
// the pattern's nodes: 16 x 16 nodes per wave, 2 x 2 waves per workgroup;
// blockIdx.y: every splits-th cell, whose partial sums the reduction adds.
// e^{2 pi i t} from a table of 64 angles (LDS) and the series of what is left,
// |x| <= pi / 64: 1e-15, a quarter of sincospi's time.
__device__ __forceinline__ void turn(double t, const double2 *table, double &cs, double &sn) {
  const double k = rint(t * 64.0);
  const double x = __builtin_fma(k, -1.0 / 64.0, t) * (2.0 * kPi), x2 = x * x;
  const double2 e = table[(int)(long long)k & 63];
  const double s =
      x * __builtin_fma(x2, __builtin_fma(x2, __builtin_fma(x2, -1.0 / 5040.0, 1.0 / 120.0), -1.0 / 6.0), 1.0);
  const double c = __builtin_fma(
      x2, __builtin_fma(x2, __builtin_fma(x2, __builtin_fma(x2, 1.0 / 40320.0, -1.0 / 720.0), 1.0 / 24.0), -0.5), 1.0);
  cs = e.x * c - e.y * s;
  sn = e.y * c + e.x * s;
}

__global__ __launch_bounds__(kT, 4) void surface_cell_cols_kernel(const SurfJob *jobs, int first) {
  __shared__ double wy[kCellMaxNodes][32];
  __shared__ double2 table[64];
  const SurfJob &jb = jobs[first + blockIdx.z];
  const SurfCells &c = jb.c;
  if (!jb.ok || c.g == 0 || (int)blockIdx.y >= jb.splits) return;
  const int nxn = c.co.fx.n, nyn = c.co.fy.n, myn = c.co.ay.n;
  const int tiles_x = (nxn + 31) / 32, bx = (int)blockIdx.x % tiles_x, by = (int)blockIdx.x / tiles_x;
  const int wave = threadIdx.x / 64, l = threadIdx.x & 63, m = l & 15, gq = l >> 4;
  const int x = bx * 32 + (wave & 1) * 16 + m, y0 = (by * 2 + (wave >> 1)) * 16;
  if (by * 32 >= nyn) return;
  for (int i = threadIdx.x; i < myn * 32; i += kT)
    wy[i / 32][i % 32] = c.co.wy[(size_t)(i / 32) * nyn + min(by * 32 + i % 32, nyn - 1)];
  if (threadIdx.x < 64) sincospi(threadIdx.x / 32.0, &table[threadIdx.x].y, &table[threadIdx.x].x);
  __syncthreads();
  if (x - m >= nxn || y0 >= nyn) return;
  const int xc = min(x, nxn - 1);
  const double *w = &wy[gq][(wave >> 1) * 16 + m], *w32 = &wy[gq][(wave >> 1) * 16 + prow(m)];
  double q[4][3], re[4] = {}, im[4] = {};
  float nr[4] = {}, ni[4] = {};
#pragma unroll
  for (int r = 0; r < 4; ++r)
    for (int k = 0; k < 3; ++k) q[r][k] = jb.sh.nodes[3 * ((size_t)xc * nyn + min(y0 + gq + 4 * r, nyn - 1)) + k];
  const int ncells = c.g * c.g * c.gz;
  for (int id = blockIdx.y; id < ncells; id += jb.splits) {
    const SurfCell &cell = c.cells[id];
    if (cell.count == 0) continue;
    const double2 *tf = c.tf + ((size_t)id * myn + gq) * nxn + xc;
    const float2 *tn = c.tn + ((size_t)id * myn + gq) * nxn + xc;
    Fields<2> acc;
    clear(acc);
#pragma unroll 4
    for (int k = 0; k < myn; k += 4) {
      const double2 v = tf[(size_t)k * nxn];
      const float2 n = tn[(size_t)k * nxn];
      const double a = w[32 * k];
      const float a32 = (float)w32[32 * k];
      acc.re = mfma64(a, v.x, acc.re);
      acc.im = mfma64(a, v.y, acc.im);
      acc.g[0] = mfma32(a32, n.x, acc.g[0]);
      acc.g[1] = mfma32(a32, n.y, acc.g[1]);
    }
    const double cx = cell.centre[0], cy = cell.centre[1], cz = cell.centre[2];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const double t = __builtin_fma(q[r][2], cz, __builtin_fma(q[r][1], cy, q[r][0] * cx));
      double sn, cs;
      turn(t - rint(t), table, cs, sn);
      re[r] += acc.re[r] * cs + acc.im[r] * sn;
      im[r] += acc.im[r] * cs - acc.re[r] * sn;
      const float cf = (float)cs, sf = (float)sn;
      nr[r] += acc.g[0][r] * cf + acc.g[1][r] * sf;
      ni[r] += acc.g[1][r] * cf - acc.g[0][r] * sf;
    }
  }
  if (x >= nxn) return;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int y = y0 + gq + 4 * r;
    if (y >= nyn) continue;
    const int node = x * nyn + y;
    if (jb.splits > 1) {  // as store_node leaves them
      const size_t o = ((size_t)(node / kT) * jb.splits + blockIdx.y) * kT + node % kT;
      jb.slot_f[o] = make_double2(re[r], -im[r]);
      jb.slot_n[o] = make_float2(ni[r] / (-2.0f * (float)kPi), nr[r] / (-2.0f * (float)kPi));
    } else {
      jb.f[node] = make_double2(re[r], im[r]);
      jb.n[node] = make_float2(nr[r], ni[r]);
    }
  }
}

// Along the rows, t[k][x] = sum_i node[i][k] tx[i][x] of F (FP64), of F with the
// weights' derivatives and of N: 16 node rows x 16 columns per wave;
// blockIdx.x: 64 columns, blockIdx.y: 16 node rows, blockIdx.z: pattern.
__global__ __launch_bounds__(kT) void surface_rows_kernel(const SurfJob *jobs, int first) {
  const SurfJob &jb = jobs[first + blockIdx.z];
  if (!jb.ok) return;
  const int nyn = jb.sh.ay.n, nxn = jb.sh.ax.n, nx = jb.nx;
  const int l = threadIdx.x & 63, m = l & 15, gq = l >> 4;
  const int k0 = (int)blockIdx.y * 16, x = (int)blockIdx.x * 64 + (int)(threadIdx.x / 64) * 16 + m;
  if (k0 >= nyn || x - m >= nx) return;
  // rows and columns past the end repeat the last one and are not stored
  const size_t row = (size_t)gq * nyn + min(k0 + m, nyn - 1), prow_ = (size_t)gq * nyn + min(k0 + prow(m), nyn - 1);
  const double2 *f = jb.f + row, *fp = jb.f + prow_;
  const float2 *n = jb.n + prow_;
  const double *tx = jb.sh.tx + (size_t)gq * nx + min(x, nx - 1);
  const float2 *tx32 = jb.sh.tx32 + (size_t)gq * nx + min(x, nx - 1);
  Fields<4> acc;
  clear(acc);
#pragma unroll 4
  for (int i = 0; i < nxn; i += 4) {
    const double2 fv = f[(size_t)i * nyn], fq = fp[(size_t)i * nyn];
    const float2 nv = n[(size_t)i * nyn];
    const double b = tx[(size_t)i * nx];
    const float2 b32 = tx32[(size_t)i * nx];
    acc.re = mfma64(fv.x, b, acc.re);
    acc.im = mfma64(fv.y, b, acc.im);
    acc.g[0] = mfma32((float)fq.x, b32.y, acc.g[0]);
    acc.g[1] = mfma32((float)fq.y, b32.y, acc.g[1]);
    acc.g[2] = mfma32(nv.x, b32.x, acc.g[2]);
    acc.g[3] = mfma32(nv.y, b32.x, acc.g[3]);
  }
  if (x >= nx) return;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int k = k0 + gq + 4 * r;
    if (k >= nyn) continue;
    const size_t o = (size_t)k * nx + x;
    jb.t64[o] = make_double2(acc.re[r], acc.im[r]);
    jb.t32[o] = make_float4(acc.g[0][r], acc.g[1][r], acc.g[2][r], acc.g[3][r]);
  }
}

// Along the columns, F(y, x) = sum_k ty[k][y] t[k][x] and its derivatives, then the
// list's deviation, the centre's phase and the intensity: 16 x 16 pixels per
// wave, 2 x 2 waves per workgroup. (Two tiles per wave, which share the operand t,
// keep two waves per SIMD instead of four: 82 us against 57 us on 1024^2 pixels
// and 188 nodes.)
__global__ __launch_bounds__(kT) void surface_cols_kernel(const SurfJob *jobs, int first, const float *__restrict__ dev,
                                                          const float *__restrict__ hkl, float2 *__restrict__ F,
                                                          float *__restrict__ I) {
  const SurfJob &jb = jobs[first + blockIdx.z];
  if (!jb.ok) return;
  const int nyn = jb.sh.ay.n, nx = jb.nx, ny = jb.ny;
  const int wave = threadIdx.x / 64, l = threadIdx.x & 63, m = l & 15, gq = l >> 4;
  const int x = (int)blockIdx.x * 32 + (wave & 1) * 16 + m, y0 = ((int)blockIdx.y * 2 + (wave >> 1)) * 16;
  if (x - m >= nx || y0 >= ny) return;
  const size_t xc = (size_t)gq * nx + min(x, nx - 1);
  const double2 *t64 = jb.t64 + xc;
  const float4 *t32 = jb.t32 + xc;
  const double *w = jb.sh.ty + (size_t)gq * ny + min(y0 + m, ny - 1);
  const float2 *w32 = jb.sh.ty32 + (size_t)gq * ny + min(y0 + prow(m), ny - 1);
  Fields<6> acc;  // F; dF/du, N, dF/dv
  clear(acc);
#pragma unroll 4
  for (int k = 0; k < nyn; k += 4) {
    const double2 v = t64[(size_t)k * nx];
    const float4 g = t32[(size_t)k * nx];
    const double a = w[(size_t)k * ny];
    const float2 a32 = w32[(size_t)k * ny];
    acc.re = mfma64(a, v.x, acc.re);
    acc.im = mfma64(a, v.y, acc.im);
    acc.g[0] = mfma32(a32.x, g.x, acc.g[0]);
    acc.g[1] = mfma32(a32.x, g.y, acc.g[1]);
    acc.g[2] = mfma32(a32.x, g.z, acc.g[2]);
    acc.g[3] = mfma32(a32.x, g.w, acc.g[3]);
    acc.g[4] = mfma32(a32.y, (float)v.x, acc.g[4]);
    acc.g[5] = mfma32(a32.y, (float)v.y, acc.g[5]);
  }
  if (x >= nx) return;
  double cx = jb.r0[0], cy = jb.r0[1], cz = jb.r0[2];
  if (jb.has_rot) {
    const double *R = jb.rot;
    const double ax = cx, ay = cy, az = cz;
    cx = __builtin_fma(R[6], az, __builtin_fma(R[3], ay, R[0] * ax));
    cy = __builtin_fma(R[7], az, __builtin_fma(R[4], ay, R[1] * ax));
    cz = __builtin_fma(R[8], az, __builtin_fma(R[5], ay, R[2] * ax));
  }
  const size_t out = (size_t)jb.pattern * ((size_t)nx * ny);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int y = y0 + gq + 4 * r;
    if (y >= ny) continue;
    const size_t p = (size_t)y * nx + x;
    const float al = dev[3 * p], be = dev[3 * p + 1], ga = dev[3 * p + 2];
    const double re =
        acc.re[r] + (double)__builtin_fmaf(ga, acc.g[2][r], __builtin_fmaf(be, acc.g[4][r], al * acc.g[0][r]));
    const double im =
        acc.im[r] + (double)__builtin_fmaf(ga, acc.g[3][r], __builtin_fmaf(be, acc.g[5][r], al * acc.g[1][r]));
    if (I) I[out + p] = (float)(re * re + im * im);
    if (F) {
      const double t = __builtin_fma((double)hkl[3 * p + 2], cz,
                                     __builtin_fma((double)hkl[3 * p + 1], cy, (double)hkl[3 * p] * cx));
      double sn, cs;
      sincospi(2.0 * __builtin_amdgcn_fract(t), &sn, &cs);
      F[out + p] = make_float2((float)(re * cs + im * sn), (float)(im * cs - re * sn));
    }
  }
}

// ---- adjoint ---------------------------------------------------------------------
//
// The gradients of a loss with dL/dI_p = g_p given need, per atom j,
//   S_j = sum_p A_p h_j(q_p),  A_p = 2 g_p F_p,  h_j(q) = f(|q|) e^{-B_j s^2} e^{2 pi i q.r_j},
// with dL/dr_j = -2 pi w_j Im sum_p q_p A_p h_j and dL/dB_j = -w_j Re sum_p s_p^2 A_p h_j
// (adjoint.hip). h_j is as smooth over the detector as F, so the transposed
// interpolation carries the pixels' values to the nodes,
//   a_v = sum_p A_p (L_v + alpha_p dL_v/du + beta_p dL_v/dv),  b_v = sum_p gamma_p A_p L_v,
// two dense products again (FP64 for A_p L_v, FP32 for the rest), and every atom
// sums nodes instead of pixels: S_j = sum_v h_j(q_v) Z_v, Z_v = a_v + 2 pi i n.r_j b_v.

// First product: t[split][k][x], sums over the split's list rows of
// ty[k][y] A + dty[k][y] beta A (t64), ty[k][y] alpha A and ty[k][y] gamma A (t32);
// 16 node rows x 16 columns per wave, blockIdx.z: rows of the list.
__global__ __launch_bounds__(kT) void surface_gather_rows_kernel(const SurfJob *job, const float2 *__restrict__ pixels,
                                                                 const float *__restrict__ dev) {
  const SurfJob &jb = *job;
  if (!jb.ok) return;
  const int nyn = jb.sh.ay.n, nx = jb.nx, ny = jb.ny;
  const int l = threadIdx.x & 63, m = l & 15, gq = l >> 4;
  const int k0 = (int)blockIdx.y * 16, x = (int)blockIdx.x * 64 + (int)(threadIdx.x / 64) * 16 + m;
  if (k0 >= nyn || x - m >= nx) return;
  const int steps = (ny + 3) / 4, splits = gridDim.z;
  const int y0 = 4 * (int)((long long)steps * blockIdx.z / splits);
  const int y1 = 4 * (int)((long long)steps * (blockIdx.z + 1) / splits);
  const int xc = min(x, nx - 1);
  const size_t row = (size_t)min(k0 + m, nyn - 1) * ny, prow_ = (size_t)min(k0 + prow(m), nyn - 1) * ny;
  const double *w = jb.sh.ty + row;
  const float2 *w32 = jb.sh.ty32 + prow_;
  Fields<6> acc;
  clear(acc);
#pragma unroll 4
  for (int y = y0; y < y1; y += 4) {
    const int yy = min(y + gq, ny - 1);
    const bool in = y + gq < ny;  // rows past the end weigh nothing
    const double a = in ? w[yy] : 0.0;
    const float2 a32 = in ? w32[yy] : make_float2(0.0f, 0.0f);
    const size_t p = (size_t)yy * nx + xc;
    const float2 v = pixels[p];
    const float al = dev[3 * p], be = dev[3 * p + 1], ga = dev[3 * p + 2];
    acc.re = mfma64(a, (double)v.x, acc.re);
    acc.im = mfma64(a, (double)v.y, acc.im);
    acc.g[0] = mfma32(a32.y, be * v.x, acc.g[0]);
    acc.g[1] = mfma32(a32.y, be * v.y, acc.g[1]);
    acc.g[2] = mfma32(a32.x, al * v.x, acc.g[2]);
    acc.g[3] = mfma32(a32.x, al * v.y, acc.g[3]);
    acc.g[4] = mfma32(a32.x, ga * v.x, acc.g[4]);
    acc.g[5] = mfma32(a32.x, ga * v.y, acc.g[5]);
  }
  if (x >= nx) return;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int k = k0 + gq + 4 * r;
    if (k >= nyn) continue;
    const size_t o = ((size_t)blockIdx.z * nyn + k) * nx + x;
    jb.t64[o] = make_double2(acc.re[r] + (double)acc.g[0][r], acc.im[r] + (double)acc.g[1][r]);
    jb.t32[o] = make_float4(acc.g[2][r], acc.g[3][r], acc.g[4][r], acc.g[5][r]);
  }
}

// Second product: a (jb.f) and b (jb.n) of the nodes (i, k) of one node row k.
// The workgroup adds the splits of 256 columns into LDS at a time; each wave then
// takes every fourth of its part's nodes, the lanes sharing the columns.
constexpr int kGatherParts = 4;  // workgroups per node row

__global__ __launch_bounds__(kT) void surface_gather_nodes_kernel(const SurfJob *job, int splits) {
  const SurfJob &jb = *job;
  if (!jb.ok) return;
  const int nyn = jb.sh.ay.n, nxn = jb.sh.ax.n, nx = jb.nx;
  const int k = blockIdx.y, part = blockIdx.x;
  if (k >= nyn) return;
  __shared__ double2 t64[kT];
  __shared__ float4 t32[kT];
  __shared__ double2 sum_a[kSurfMaxNodes / kGatherParts + 4];
  __shared__ float2 sum_b[kSurfMaxNodes / kGatherParts + 4];
  const int i0 = nxn * part / kGatherParts, i1 = nxn * (part + 1) / kGatherParts;
  const int t = threadIdx.x, lane = t & 63, wave = t / 64;
  for (int x0 = 0; x0 < nx; x0 += kT) {
    double2 a = make_double2(0.0, 0.0);
    float4 g = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (x0 + t < nx) {
#pragma unroll 8
      for (int s = 0; s < splits; ++s) {
        const size_t o = ((size_t)s * nyn + k) * nx + x0 + t;
        const double2 v = jb.t64[o];
        const float4 h = jb.t32[o];
        a.x += v.x;
        a.y += v.y;
        g.x += h.x;
        g.y += h.y;
        g.z += h.z;
        g.w += h.w;
      }
    }
    __syncthreads();
    t64[t] = a;
    t32[t] = g;
    __syncthreads();
    for (int i = i0 + wave; i < i1; i += kT / 64) {
      double re = 0.0, im = 0.0;
      float br = 0.0f, bi = 0.0f;
#pragma unroll
      for (int c = 0; c < kT / 64; ++c) {
        const int xl = c * 64 + lane, x = min(x0 + xl, nx - 1);  // columns past the end hold zeros
        const double w = jb.sh.tx[(size_t)i * nx + x];
        const float2 w32 = jb.sh.tx32[(size_t)i * nx + x];
        const double2 v = t64[xl];
        const float4 h = t32[xl];
        re = __builtin_fma(w, v.x, re + (double)(w32.y * h.x));
        im = __builtin_fma(w, v.y, im + (double)(w32.y * h.y));
        br = __builtin_fmaf(w32.x, h.z, br);
        bi = __builtin_fmaf(w32.x, h.w, bi);
      }
      for (int o = 32; o > 0; o >>= 1) {
        re += __shfl_xor(re, o);
        im += __shfl_xor(im, o);
        br += __shfl_xor(br, o);
        bi += __shfl_xor(bi, o);
      }
      if (lane == 0) {
        if (x0 == 0) {
          sum_a[i - i0] = make_double2(re, im);
          sum_b[i - i0] = make_float2(br, bi);
        } else {
          sum_a[i - i0].x += re;
          sum_a[i - i0].y += im;
          sum_b[i - i0].x += br;
          sum_b[i - i0].y += bi;
        }
      }
    }
  }
  __syncthreads();
  for (int i = i0 + t; i < i1; i += kT) {
    jb.f[(size_t)i * nyn + k] = sum_a[i - i0];
    jb.n[(size_t)i * nyn + k] = sum_b[i - i0];
  }
}

// A node as every atom of one species reads it: f(|q|) a, 2 pi f(|q|) b.
struct __align__(16) AdjNode {
  double qx, qy, qz;
  float ar, ai, br, bi;
  float qxf, qyf, qzf;
  float s2, nl2, pad;
};
static_assert(sizeof(AdjNode) == 64, "adjoint node record");

// Per atom: U = Im sum q h Z and V = Re sum s^2 h Z over a range of nodes; one
// tile of 512 atoms of one species per workgroup (2 per lane), the nodes
// staged in LDS 128 at a time. Per term 3 FP64 FMAs, a fraction and a conversion,
// a sine and cosine, and 8 FP32 FMAs (with B an exponential and 2 more). FP32 sums over a chunk, FP64 across chunks.
template <bool HAS_B, bool WANT_B>
__global__ __launch_bounds__(kT) void surface_adjoint_kernel(const SurfJob *job, const SurfAtomTile *tiles,
                                                             const float *__restrict__ ff, float b_global,
                                                             double4 *__restrict__ partial) {
  constexpr int KA = kSurfAtomsPerLane, kChunk = 128;
  __shared__ AdjNode sm[kChunk];
  const SurfJob &jb = *job;
  if (!jb.ok) return;
  const SurfAtomTile tile = tiles[blockIdx.x];
  const int nodes = jb.sh.ax.n * jb.sh.ay.n, split = blockIdx.y, nsplit = gridDim.y;
  const int n_begin = (int)((long long)nodes * split / nsplit), n_end = (int)((long long)nodes * (split + 1) / nsplit);
  const float Bs = tile.species == SPSIM_HIP_UNIT_SPECIES ? 0.0f : b_global;
  const float *c = ff + tile.species * SPSIM_HIP_FF_STRIDE;
  double rx[KA], ry[KA], rz[KA], Ux[KA], Uy[KA], Uz[KA], V[KA];
  float nr[KA], bj[KA];
#pragma unroll
  for (int k = 0; k < KA; ++k) {
    const int i = threadIdx.x + k * kT;
    const bool ok = i < tile.count;
    const spsim_hip_atom at = ok ? jb.atoms[tile.start + i] : spsim_hip_atom{0.f, 0.f, 0.f, 0.f};
    rx[k] = ok ? at.x - jb.r0[0] : 0.0;
    ry[k] = ok ? at.y - jb.r0[1] : 0.0;
    rz[k] = ok ? at.z - jb.r0[2] : 0.0;
    nr[k] = jb.normal[0] * (float)rx[k] + jb.normal[1] * (float)ry[k] + jb.normal[2] * (float)rz[k];
    bj[k] = (HAS_B && ok) ? jb.atom_b[tile.start + i] : 0.0f;
    Ux[k] = Uy[k] = Uz[k] = V[k] = 0.0;
  }
  for (int n0 = n_begin; n0 < n_end; n0 += kChunk) {
    const int n = min(kChunk, n_end - n0);
    __syncthreads();
    if ((int)threadIdx.x < n) {
      const size_t node = n0 + threadIdx.x;
      const double *q = jb.sh.nodes + 3 * node;
      AdjNode r;
      r.qx = q[0];
      r.qy = q[1];
      r.qz = q[2];
      r.qxf = (float)q[0];
      r.qyf = (float)q[1];
      r.qzf = (float)q[2];
      const double s2 = (q[0] * q[0] + q[1] * q[1] + q[2] * q[2]) * 2.5e-21;
      const double f = (1.0 + kTrigBias) * form_factor64(c, s2, Bs);
      const double2 a = jb.f[node];
      r.ar = (float)(f * a.x);
      r.ai = (float)(f * a.y);
      const float2 b = jb.n[node];
      r.br = (float)(2.0 * kPi * f) * b.x;
      r.bi = (float)(2.0 * kPi * f) * b.y;
      r.s2 = (float)s2;
      r.nl2 = (float)(-s2 * kLog2e);
      r.pad = 0.0f;
      sm[threadIdx.x] = r;
    }
    __syncthreads();
    float ux[KA], uy[KA], uz[KA], v[KA];
#pragma unroll
    for (int k = 0; k < KA; ++k) ux[k] = uy[k] = uz[k] = v[k] = 0.0f;
    for (int i = 0; i < n; ++i) {
      const AdjNode r = sm[i];
#pragma unroll
      for (int k = 0; k < KA; ++k) {
        const double t = __builtin_fma(r.qz, rz[k], __builtin_fma(r.qy, ry[k], r.qx * rx[k]));
        const float ph = (float)__builtin_amdgcn_fract(t);
        float cs = __builtin_amdgcn_cosf(ph), sn = __builtin_amdgcn_sinf(ph);
        if constexpr (HAS_B) {
          const float e = __builtin_amdgcn_exp2f(bj[k] * r.nl2);
          cs *= e;
          sn *= e;
        }
        // Z = a + i (2 pi n.r b)
        const float zr = __builtin_fmaf(-nr[k], r.bi, r.ar);
        const float zi = __builtin_fmaf(nr[k], r.br, r.ai);
        const float u = __builtin_fmaf(cs, zi, sn * zr);
        ux[k] = __builtin_fmaf(u, r.qxf, ux[k]);
        uy[k] = __builtin_fmaf(u, r.qyf, uy[k]);
        uz[k] = __builtin_fmaf(u, r.qzf, uz[k]);
        if constexpr (WANT_B) v[k] = __builtin_fmaf(r.s2, __builtin_fmaf(cs, zr, -(sn * zi)), v[k]);
      }
    }
#pragma unroll
    for (int k = 0; k < KA; ++k) {
      Ux[k] += ux[k];
      Uy[k] += uy[k];
      Uz[k] += uz[k];
      V[k] += v[k];
    }
  }
#pragma unroll
  for (int k = 0; k < KA; ++k) {
    const int i = threadIdx.x + k * kT;
    if (i < tile.count)
      partial[(size_t)split * jb.natoms + tile.start + i] = make_double4(Ux[k], Uy[k], Uz[k], V[k]);
  }
}

size_t align_up(size_t n) { return (n + 255) / 256 * 256; }

// Row ranges of the adjoint's first product: enough waves for the chip.
int gather_splits(int nx) { return std::max(2, std::min(8, 4096 / nx)); }

// A tiling's slots beyond the nodes: an octant grid's diagonals and its last tile.
constexpr int kSlotSlack = 2 * kSurfMaxNodes + 8 * kT;

// Workspace of one pattern: the nodes of an axis are limited to what can pay
// (worth() needs n_x n_y below about a third of the pixels).
struct SingleLayout {
  int max_nx, max_ny, slot_cap;
  size_t fit, records, centres, job, dev, nodes, tx, ty, tx32, ty32, prep, f, n, slot_f, slot_n, t64, t32, total;
  // sums by cells, for large patterns (not of spectra)
  int cells;
  long long cell_sums, cell_rows;
  size_t c_nodes, c_wx, c_wy, c_id, c_sorted, c_cells, c_segs, c_range, c_order, c_f, c_n, c_tf, c_tn;
};

// Terms below which no pattern's node sums take long enough for cells (100 us:
// 50,000 atoms at 80^2 nodes, on 512^2 pixels), so that their launches are left out.
constexpr long long kCellMinTerms = 10000000000;
// Ranges and cells hold at most these for one pattern.
constexpr long long kCellSums = 4 << 20, kCellRows = 4 << 20;

SingleLayout single_layout(int nx, int ny, int natoms, int nsegs, SurfKind kind) {
  const bool adjoint = kind == SurfKind::kAdjoint;
  SingleLayout l;
  auto cap = [](int n) { return std::max(kSurfMinNodes, std::min(kSurfMaxNodes, (int)(0.6 * n) / 4 * 4)); };
  l.max_nx = cap(nx);
  l.max_ny = cap(ny);
  const size_t nodes = (size_t)l.max_nx * l.max_ny, npix = (size_t)nx * ny;
  l.slot_cap = std::max(1 << 20, (int)nodes + kSlotSlack);
  size_t at = 0;
  auto take = [&](size_t bytes) {
    const size_t o = at;
    at += align_up(bytes);
    return o;
  };
  l.job = take(sizeof(SurfJob));
  l.fit = take(sizeof(SurfFit));
  l.records = take(sizeof(SurfRecord) * (kSurfListBlocks + kSurfAtomBlocks));
  l.centres = take(sizeof(double) * 3);
  l.dev = take(sizeof(float) * 3 * npix);
  l.nodes = take(sizeof(double) * 3 * nodes);
  l.tx = take(sizeof(double) * (size_t)l.max_nx * nx);
  l.ty = take(sizeof(double) * (size_t)l.max_ny * ny);
  l.tx32 = take(sizeof(float2) * (size_t)l.max_nx * nx);
  l.ty32 = take(sizeof(float2) * (size_t)l.max_ny * ny);
  l.prep = adjoint ? take(sizeof(float2) * npix) : take(sizeof(NodeAtom) * (size_t)natoms);
  l.f = take(sizeof(double2) * nodes);
  l.n = take(sizeof(float2) * nodes);
  const size_t rows = (size_t)l.max_ny * nx * (adjoint ? gather_splits(nx) : 1);
  l.slot_f = take(adjoint ? 0 : sizeof(double2) * (size_t)l.slot_cap);
  l.slot_n = take(adjoint ? 0 : sizeof(float2) * (size_t)l.slot_cap);
  l.t64 = take(sizeof(double2) * rows);
  l.t32 = take(sizeof(float4) * rows);
  l.cells = kind == SurfKind::kSum && (long long)npix * natoms >= kCellMinTerms ? kMaxCells : 0;
  l.cell_sums = l.cell_rows = 0;
  if (l.cells > 0) {
    l.cell_sums = kCellSums;
    l.cell_rows = kCellRows;
    l.c_nodes = take(sizeof(double) * 3 * kCellMaxNodes * kCellMaxNodes);
    l.c_wx = take(sizeof(double) * kCellMaxNodes * (size_t)l.max_nx);
    l.c_wy = take(sizeof(double) * kCellMaxNodes * (size_t)l.max_ny);
    l.c_id = take(sizeof(unsigned short) * ((size_t)natoms + 8));
    l.c_sorted = take(sizeof(NodeAtom) * (size_t)natoms);
    l.c_cells = take(sizeof(SurfCell) * kMaxCells);
    l.c_segs = take(sizeof(spsim_hip_segment) * kMaxCells * (size_t)nsegs);
    l.c_range = take(sizeof(int) * (512 + kMaxCells + 1));
    l.c_order = take(sizeof(int) * (size_t)natoms);
    l.c_f = take(sizeof(double2) * (size_t)l.cell_sums);
    l.c_n = take(sizeof(float2) * (size_t)l.cell_sums);
    l.c_tf = take(sizeof(double2) * (size_t)l.cell_rows);
    l.c_tn = take(sizeof(float2) * (size_t)l.cell_rows);
  }
  l.total = at;
  return l;
}

void launch_interpolation(const SurfJob *jobs, int first, int count, int nx, int ny, int max_nodes, int max_ny,
                          const float *dev, const float *hkl, float2 *F, float *I, hipStream_t s) {
  if (max_nodes > 0)  // some pattern's atoms are split
    hipLaunchKernelGGL(surface_reduce_kernel, dim3((max_nodes + kSlotSlack + kT - 1) / kT, 2, count), dim3(kT), 0, s,
                       jobs, first);
  hipLaunchKernelGGL(surface_rows_kernel, dim3((nx + 63) / 64, (max_ny + 15) / 16, count), dim3(kT), 0, s, jobs,
                     first);
  hipLaunchKernelGGL(surface_cols_kernel, dim3((nx + 31) / 32, (ny + 31) / 32, count), dim3(kT), 0, s, jobs, first, dev,
                     hkl, F, I);
}

// Grid sizes for the sums by cells of some patterns.
struct CellBounds {
  int cells;        // per pattern
  long long items;  // (range, tile) pairs
  int rows;         // workgroups of the first product
  int nxn, nyn, splits;
};

void launch_cells(const SurfJob *jobs, int first, int count, const CellBounds &b, const float *ff, float b_global,
                  bool has_b, hipStream_t s) {
  hipLaunchKernelGGL(surface_sort_kernel, dim3(b.cells, 1, count), dim3(kSortT), 0, s, jobs, first);
  hipLaunchKernelGGL(has_b ? surface_cell_nodes_kernel<true> : surface_cell_nodes_kernel<false>,
                     dim3((unsigned)b.items, count), dim3(kT), 0, s, jobs, first, ff, b_global);
  hipLaunchKernelGGL(surface_cell_rows_kernel, dim3(b.rows, count), dim3(kT), 0, s, jobs, first);
  hipLaunchKernelGGL(surface_cell_cols_kernel, dim3(((b.nxn + 31) / 32) * ((b.nyn + 31) / 32), b.splits, count),
                     dim3(kT), 0, s, jobs, first);
}

// Bound on how much a matrix lengthens a vector: the root of the largest
// absolute row sum of R^T R (Gershgorin). 1 for a rotation, but callers may
// pass any matrix; infinite where an element is not finite.
double rotation_norm(const double *R) {
  double most = 0.0;
  for (int i = 0; i < 3; ++i) {
    double row = 0.0;
    for (int j = 0; j < 3; ++j) row += std::fabs(R[i] * R[j] + R[3 + i] * R[3 + j] + R[6 + i] * R[6 + j]);
    if (!std::isfinite(row)) return INFINITY;
    most = std::max(most, row);
  }
  return std::sqrt(most);
}

const void *nodes_kernel(bool has_b, bool spec) {
  if (spec)
    return has_b ? (const void *)&surface_nodes_kernel<true, true> : (const void *)&surface_nodes_kernel<false, true>;
  return has_b ? (const void *)&surface_nodes_kernel<true, false> : (const void *)&surface_nodes_kernel<false, false>;
}

int launch_nodes(const SurfJob *jobs, const SurfItem *items, int nitems, int blocks, const float *ff, float b_global,
                 bool has_b, const Spectrum *sp, hipStream_t s) {
  NoSpectrum none;
  void *params[] = {(void *)&jobs, (void *)&items,    (void *)&nitems,
                    (void *)&ff,   (void *)&b_global, sp ? (void *)sp : (void *)&none};
  SPSIM_HIP_TRY(hipLaunchKernel(nodes_kernel(has_b, sp != nullptr), dim3(blocks), dim3(kT), params, 0, s));
  return SPSIM_HIP_OK;
}

}  // namespace

bool surf_worth(long long nx, long long ny, long long natoms, long long min_terms) {
  return nx >= kSurfMinSide && ny >= kSurfMinSide && nx * ny * natoms >= min_terms;
}

size_t surf_single_bytes(int nx, int ny, int natoms, int nsegs, bool spectrum) {
  return single_layout(nx, ny, natoms, nsegs, spectrum ? SurfKind::kSpectrum : SurfKind::kSum).total;
}

namespace {

// Scan and plan of one pattern; the job is left at the workspace's start.
int launch_plan(const PatternLaunch &a, int nx, int ny, const Spectrum *sp, SurfKind kind, const float *gI,
                const SingleLayout &l, char *w, int slots, int cus, hipStream_t s) {
  PlanArgs p{};
  p.job.nx = nx;
  p.job.ny = ny;
  p.job.sh.nodes = (double *)(w + l.nodes);
  p.job.sh.tx = (double *)(w + l.tx);
  p.job.sh.ty = (double *)(w + l.ty);
  p.job.sh.tx32 = (float2 *)(w + l.tx32);
  p.job.sh.ty32 = (float2 *)(w + l.ty32);
  p.job.atoms = a.atoms;
  p.job.atom_b = a.atom_b;
  p.job.segs = a.segs;
  p.job.nsegs = a.nsegs;
  p.job.natoms = a.natoms;
  p.job.has_rot = a.has_rot;
  std::copy(a.rot.r, a.rot.r + 9, p.job.rot);
  p.job.f = (double2 *)(w + l.f);
  p.job.n = (float2 *)(w + l.n);
  p.job.slot_f = (double2 *)(w + l.slot_f);
  p.job.slot_n = (float2 *)(w + l.slot_n);
  p.job.prep = w + l.prep;
  p.job.t64 = (double2 *)(w + l.t64);
  p.job.t32 = (float4 *)(w + l.t32);
  p.fit = (const SurfFit *)(w + l.fit);
  p.records = (const SurfRecord *)(w + l.records);
  p.list_blocks = std::min(kSurfListBlocks, ny + 2);
  p.centres = (const double *)(w + l.centres);
  p.ff = a.ff;
  p.b_global = a.b_global;
  p.has_b = a.atom_b != nullptr;
  p.slots = slots;
  p.slot_cap = l.slot_cap;
  p.max_nx = l.max_nx;
  p.max_ny = l.max_ny;
  const bool cells = l.cells > 0;
  if (cells) {
    p.max_cells = l.cells;
    p.max_cell_sums = l.cell_sums;
    p.max_cell_rows = l.cell_rows;
    SurfCells &c = p.job.c;
    c.co.nodes = (double *)(w + l.c_nodes);
    c.co.wx = (double *)(w + l.c_wx);
    c.co.wy = (double *)(w + l.c_wy);
    c.id = (unsigned short *)(w + l.c_id);
    c.sorted = w + l.c_sorted;
    c.cells = (SurfCell *)(w + l.c_cells);
    c.segs = (spsim_hip_segment *)(w + l.c_segs);
    c.range_cell = (int *)(w + l.c_range);
    c.order = (int *)(w + l.c_order);
    c.f = (double2 *)(w + l.c_f);
    c.n = (float2 *)(w + l.c_n);
    c.tf = (double2 *)(w + l.c_tf);
    c.tn = (float2 *)(w + l.c_tn);
  }
  p.kind = kind;
  const double norm = a.has_rot ? rotation_norm(a.rot.r) : 1.0;
  p.scale = norm;
  if (sp) {
    p.scale = 0.0;
    for (int k = 0; k < sp->n; ++k) {
      p.scale = std::max(p.scale, norm * std::fabs(sp->s[k]));
      p.spread = std::max(p.spread, std::fabs(sp->s[k] / sp->sc - 1.0));
    }
  }
  p.out = (SurfJob *)(w + l.job);
  if (kind == SurfKind::kAdjoint) {
    p.hkl = a.hkl;
    p.F = a.F;
    p.gI = gI;
    p.pixels = (float2 *)(w + l.prep);
  }
  const ScanArgs sc{a.hkl,
                    nx,
                    ny,
                    p.list_blocks,
                    a.atoms,
                    a.atom_b,
                    nullptr,
                    MolInfo{0, a.natoms, 0, a.nsegs},
                    !sp,
                    (SurfFit *)(w + l.fit),
                    (float *)(w + l.dev),
                    (SurfRecord *)(w + l.records),
                    (double *)(w + l.centres)};
  hipLaunchKernelGGL(surface_scan_kernel, dim3(p.list_blocks + kSurfAtomBlocks), dim3(kT), 0, s, sc);
  hipLaunchKernelGGL(surface_plan_kernel, dim3(std::max(1, cells ? 3 * cus / 5 : 2 * cus / 3), cells ? 5 : 3), dim3(kT), 0, s, p);
  SPSIM_HIP_TRY(hipGetLastError());
  return SPSIM_HIP_OK;
}

}  // namespace

int launch_surface(const PatternLaunch &a, int nx, int ny, const Spectrum *sp, int cus, void *ws, const int **ok_flag,
                   hipStream_t s) {
  const SurfKind kind = sp ? SurfKind::kSpectrum : SurfKind::kSum;
  const SingleLayout l = single_layout(nx, ny, a.natoms, a.nsegs, kind);
  char *w = (char *)ws;
  const SurfJob *job = (const SurfJob *)(w + l.job);
  const bool has_b = a.atom_b != nullptr;
  const int slots = resident_slots(nodes_kernel(has_b, sp != nullptr), cus);
  SPSIM_TRY(launch_plan(a, nx, ny, sp, kind, nullptr, l, w, slots, cus, s));
  SPSIM_TRY(launch_nodes(job, nullptr, 0, slots, a.ff, a.b_global, has_b, sp, s));
  if (l.cells > 0) {
    CellBounds b{};
    b.cells = l.cells;
    // ranges x ceil(nodes / 128) tiles of at most cell_sums range nodes
    b.items = std::min(512 + l.cells + l.cell_sums / 128, 16LL * cus);
    b.rows = 8 * cus;
    b.nxn = l.max_nx;
    b.nyn = l.max_ny;
    b.splits = 32;
    launch_cells(job, 0, 1, b, a.ff, a.b_global, has_b, s);
  }
  launch_interpolation(job, 0, 1, nx, ny, l.max_nx * l.max_ny, l.max_ny, (const float *)(w + l.dev), a.hkl, a.F, a.I,
                       s);
  SPSIM_HIP_TRY(hipGetLastError());
  *ok_flag = &job->ok;
  return SPSIM_HIP_OK;
}

size_t surf_adjoint_bytes(int nx, int ny, int natoms) {
  return single_layout(nx, ny, natoms, 0, SurfKind::kAdjoint).total;
}

int launch_surface_adjoint(const PatternLaunch &a, const float *gI, int nx, int ny, const SurfAtomTile *tiles,
                           int ntiles, int splits, bool want_b, double4 *partial, int cus, void *ws,
                           const int **ok_flag, hipStream_t s) {
  const SingleLayout l = single_layout(nx, ny, a.natoms, 0, SurfKind::kAdjoint);
  char *w = (char *)ws;
  const SurfJob *job = (const SurfJob *)(w + l.job);
  SPSIM_TRY(launch_plan(a, nx, ny, nullptr, SurfKind::kAdjoint, gI, l, w, cus, cus, s));
  const int gs = gather_splits(nx);
  hipLaunchKernelGGL(surface_gather_rows_kernel, dim3((nx + 63) / 64, (l.max_ny + 15) / 16, gs), dim3(kT), 0, s, job,
                     (const float2 *)(w + l.prep), (const float *)(w + l.dev));
  hipLaunchKernelGGL(surface_gather_nodes_kernel, dim3(kGatherParts, l.max_ny), dim3(kT), 0, s, job, gs);
  const bool hb = a.atom_b != nullptr;
  const void *k = hb ? (want_b ? (const void *)&surface_adjoint_kernel<true, true>
                               : (const void *)&surface_adjoint_kernel<true, false>)
                     : (want_b ? (const void *)&surface_adjoint_kernel<false, true>
                               : (const void *)&surface_adjoint_kernel<false, false>);
  const float *ff = a.ff;
  float bg = a.b_global;
  void *params[] = {(void *)&job, (void *)&tiles, (void *)&ff, (void *)&bg, (void *)&partial};
  SPSIM_HIP_TRY(hipLaunchKernel(k, dim3(ntiles, splits), dim3(kT), params, 0, s));
  *ok_flag = &job->ok;
  return SPSIM_HIP_OK;
}

// ---- plans --------------------------------------------------------------------

struct SurfPlan {
  // Patterns that run together and share the workspace.
  struct Group {
    int first, count, item_first, nitems, max_nodes, max_ny, max_atoms;
    bool split;
    int celled;  // the first ones, summed by cells
    CellBounds cells;
  };
  SurfInput in{};
  std::vector<char> takes;
  std::vector<Group> groups;
  std::vector<SurfShape> shapes;
  std::vector<SurfCoarse> coarse;
  std::vector<SurfJob> jobs;
  std::vector<SurfItem> items;
  std::vector<char> image;  // of the upload
  // device memory: shapes, coarse nodes, jobs and items (one upload), the tables, the workspace
  size_t at_coarse = 0, at_jobs = 0, at_items = 0, at_tables = 0, at_ws = 0, bytes = 0;
  const SurfJob *d_jobs = nullptr;
  const SurfItem *d_items = nullptr;
  const float *dev = nullptr;
  std::vector<void *> owned;
};

namespace {

constexpr size_t kGroupBytes = (size_t)256 << 20;  // workspace of a group: about the last-level cache

__global__ __launch_bounds__(kT) void surface_prepare_kernel(const SurfJob *jobs, int first, bool has_b) {
  prepare_atoms(jobs[first + blockIdx.y], has_b, (int)(blockIdx.x * kT + threadIdx.x), (int)gridDim.x * kT);
}

// Lays the job's buffers out in a workspace from `at` on; returns the end.
size_t place(SurfJob *j, int nx, char *ws, size_t at) {
  const size_t nodes = (size_t)j->sh.ax.n * j->sh.ay.n;
  auto take = [&](size_t bytes) {
    char *p = ws + at;
    at += align_up(bytes);
    return p;
  };
  j->prep = take(sizeof(NodeAtom) * (size_t)j->natoms);
  j->f = (double2 *)take(sizeof(double2) * nodes);
  j->n = (float2 *)take(sizeof(float2) * nodes);
  const size_t slots = j->splits > 1 ? (size_t)j->tiles * j->per_lane * kT * j->splits : 0;
  j->slot_f = (double2 *)take(sizeof(double2) * slots);
  j->slot_n = (float2 *)take(sizeof(float2) * slots);
  j->t64 = (double2 *)take(sizeof(double2) * (size_t)j->sh.ay.n * nx);
  j->t32 = (float4 *)take(sizeof(float4) * (size_t)j->sh.ay.n * nx);
  if (j->c.g > 0) {
    SurfCells &c = j->c;
    const size_t cells = (size_t)c.g * c.g * c.gz, ranges = j->natoms / cell_range(j->natoms) + cells;
    const size_t sums = ranges * c.co.ax.n * c.co.ay.n, rows = cells * c.co.ay.n * j->sh.ax.n;
    c.id = (unsigned short *)take(sizeof(unsigned short) * ((size_t)j->natoms + 8));
    c.order = (int *)take(sizeof(int) * (size_t)j->natoms);
    c.sorted = take(sizeof(NodeAtom) * (size_t)j->natoms);
    c.cells = (SurfCell *)take(sizeof(SurfCell) * cells);
    c.segs = (spsim_hip_segment *)take(sizeof(spsim_hip_segment) * cells * j->nsegs);
    c.range_cell = (int *)take(sizeof(int) * ranges);
    c.f = (double2 *)take(sizeof(double2) * sums);
    c.n = (float2 *)take(sizeof(float2) * sums);
    c.tf = (double2 *)take(sizeof(double2) * rows);
    c.tn = (float2 *)take(sizeof(float2) * rows);
  }
  return at;
}

// The same for a shape's node positions and weights.
size_t place_tables(SurfShape *sh, int nx, int ny, char *mem, size_t at) {
  auto take = [&](size_t bytes) {
    char *p = mem + at;
    at += align_up(bytes);
    return p;
  };
  const size_t wx = (size_t)sh->ax.n * nx, wy = (size_t)sh->ay.n * ny;
  sh->nodes = (double *)take(sizeof(double) * 3 * sh->ax.n * sh->ay.n);
  sh->tx = (double *)take(sizeof(double) * wx);
  sh->ty = (double *)take(sizeof(double) * wy);
  sh->tx32 = (float2 *)take(sizeof(float2) * wx);
  sh->ty32 = (float2 *)take(sizeof(float2) * wy);
  return at;
}

size_t place_tables(SurfCoarse *co, char *mem, size_t at) {
  auto take = [&](size_t bytes) {
    char *p = mem + at;
    at += align_up(bytes);
    return p;
  };
  co->nodes = (double *)take(sizeof(double) * 3 * co->ax.n * co->ay.n);
  co->wx = (double *)take(sizeof(double) * (size_t)co->ax.n * co->fx.n);
  co->wy = (double *)take(sizeof(double) * (size_t)co->ay.n * co->fy.n);
  return at;
}

// Issue cycles of one atom in a lane's nodes (node_tiling).
double lane_cost(int per_lane) { return per_lane == 8 ? 321.0 : (per_lane == 1 ? 75.0 : 57.0 * per_lane); }

// Issue cycles of a pattern's interpolation: 85 us on 1024^2 pixels at 188 nodes.
double interpolation_cost(double nodes_x, double nodes_y, double nx, double ny) {
  return 57.0 * (nx * ny * nodes_y + nx * nodes_x * nodes_y);
}

// Splits a group's atoms so that its work items number about four per resident
// workgroup, and appends the items, largest first.
void split_group(std::vector<SurfJob> &jobs, int first, int count, int slots, std::vector<SurfItem> *items) {
  double work = 0.0;
  for (int i = first; i < first + count; ++i)
    if (jobs[i].c.g == 0) work += (double)jobs[i].tiles * lane_cost(jobs[i].per_lane) * jobs[i].natoms;
  const double share = std::max(work / (4.0 * slots), 128.0 * lane_cost(4));
  const size_t begin = items->size();
  for (int i = first; i < first + count; ++i) {
    SurfJob &j = jobs[i];
    if (j.c.g > 0) continue;  // summed by cells
    j.splits = std::max(1, std::min(kSurfMaxSplits, (int)std::ceil(lane_cost(j.per_lane) * j.natoms / share)));
    for (int t = 0; t < j.tiles; ++t)
      for (int k = 0; k < j.splits; ++k) items->push_back(SurfItem{i, t, k, 0});
  }
  std::stable_sort(items->begin() + begin, items->end(), [&](const SurfItem &a, const SurfItem &b) {
    const SurfJob &x = jobs[a.job], &y = jobs[b.job];
    return lane_cost(x.per_lane) * x.natoms / x.splits > lane_cost(y.per_lane) * y.natoms / y.splits;
  });
}

// Scan memory, within a block of surf_scan_bytes.
struct ScanLayout {
  size_t fit, dev, records, centres, total;
  int list_blocks;
};
ScanLayout scan_layout(int nx, int ny, int nmol) {
  ScanLayout l{};
  l.list_blocks = std::min(kSurfListBlocks, ny + 2);
  size_t at = 0;
  auto take = [&](size_t bytes) {
    const size_t o = at;
    at += align_up(bytes);
    return o;
  };
  l.fit = take(sizeof(SurfFit));
  l.dev = take(sizeof(float) * 3 * (size_t)nx * ny);
  l.records = take(sizeof(SurfRecord) * (l.list_blocks + (size_t)nmol * kSurfAtomBlocks));
  l.centres = take(sizeof(double) * 3 * (size_t)nmol);
  l.total = at;
  return l;
}

// Node counts of an axis: multiples of 4 up to 64 and of 8 from there on, so
// that molecules of similar size share their tables; the need falls as the
// count grows and the stretch with it.
int axis_count(int k) { return k <= 12 ? kSurfMinNodes + 4 * k : 64 + 8 * (k - 12); }

// An axis with the largest slope times density of the counts that were asked for
// (negative: not yet).
struct AxisSlopes {
  explicit AxisSlopes(const SurfSlopes &s) : slope(s) { std::fill(steepest, steepest + kSurfMaxNodes / 4 + 1, -1.0f); }
  const SurfSlopes &slope;
  float steepest[kSurfMaxNodes / 4 + 1];
};

// Whether n nodes (a multiple of 4) are enough: axis_need() with the densities of
// every count formed once.
bool enough_nodes(AxisSlopes &axis, float radius, const float *h, float b, int n) {
  struct Line {
    float as, density[kLines];
  };
  static const std::vector<Line> lines = [] {
    std::vector<Line> l(kSurfMaxNodes / 4 + 1);
    for (int i = 1; i <= kSurfMaxNodes / 4; ++i) {
      const float a = axis_stretch(4 * i);
      l[i].as = std::asin(a);
      for (int k = 0; k < kLines; ++k) l[i].density[k] = line_density(k, a, l[i].as);
    }
    return l;
  }();
  const Line &l = lines[n / 4];
  float &steepest = axis.steepest[n / 4];
  if (steepest < 0.0f)
    for (int k = 0; k < kLines; ++k) steepest = std::max(steepest, axis.slope.all[k] * l.density[k]);
  return axis_need(axis.slope, radius, h, b, l.as, [&](int k) { return l.density[k]; }, [&] { return steepest; }) <= (float)n;
}

int axis_nodes(AxisSlopes &axis, double radius, float b) {
  const float r = (float)radius, h[3] = {r, r, r};
  int lo = -1, hi = 12 + (kSurfMaxNodes - 64) / 8;
  if (!enough_nodes(axis, r, h, b, axis_count(hi))) return 0;
  while (hi - lo > 1) {
    const int mid = (lo + hi) / 2;
    (enough_nodes(axis, r, h, b, axis_count(mid)) ? hi : lo) = mid;
  }
  return axis_count(hi);
}

// The same for a box of half edges h, in multiples of 4 up to kCellMaxNodes.
int box_nodes(AxisSlopes &axis, const float *h, float b) {
  const float r = std::sqrt(h[0] * h[0] + h[1] * h[1] + h[2] * h[2]);
  int lo = -1, hi = (kCellMaxNodes - kCellMinNodes) / 4;
  if (!enough_nodes(axis, r, h, b, kCellMaxNodes)) return 0;
  while (hi - lo > 1) {
    const int mid = (lo + hi) / 2;
    (enough_nodes(axis, r, h, b, kCellMinNodes + 4 * mid) ? hi : lo) = mid;
  }
  return kCellMinNodes + 4 * hi;
}

// How a molecule's patterns are evaluated: their nodes and cells, if any.
struct Choice {
  double norm = -1.0;  // of the matrices it holds for
  bool taken = false;
  SurfAxis ax{}, ay{};
  int g = 0, gz = 0, mx = 0, my = 0;
  int shape = -1, coarse = -1;
};

SurfAxis axis_of(int n) {
  SurfAxis a{n, axis_stretch(n), 0.0};
  a.asin_a = std::asin(a.a);
  return a;
}

Choice choose(const SurfHead &head, AxisSlopes &along_x, AxisSlopes &along_y, SurfMol mol, double norm, int nx, int ny,
              int natoms, const double *limit) {
  Choice c;
  c.norm = norm;
  mol.radius *= norm;
  if (natoms <= 0 || !smooth(mol, head.s2max)) return c;
  const float b = mol.b_smooth;
  const int n[2] = {axis_nodes(along_x, mol.radius, b), axis_nodes(along_y, mol.radius, b)};
  if (n[0] == 0 || n[1] == 0) return c;
  c.ax = axis_of(n[0]);
  c.ay = axis_of(n[1]);
  const bool octants = head.sym == 2 && n[0] == n[1];
  int per_lane, tiles;
  double sums = sums_cost(n[0], n[1], octants, natoms, &per_lane, &tiles);
  // cells: the launches are shared by a plan's patterns
  double least = 0.7 * sums - 1e9;
  for (int k = 0; k < kCellGrids && mol.ordered && least > 0.0; ++k) {
    int g, gz;
    cell_grid(k, &g, &gz);
    const float r = (float)mol.radius, h[3] = {r / g, r / g, r / gz};
    const int mx = box_nodes(along_x, h, b), my = box_nodes(along_y, h, b);
    if (mx == 0 || my == 0 || (long long)(natoms / cell_range(natoms) + g * g * gz) * mx * my > kCellSums ||
        (long long)g * g * gz * my * n[0] > kCellRows)
      continue;
    const double cost = cells_cost(n[0], n[1], mx, my, g * g * gz, octants && mx == my, natoms);
    if (cost >= least) continue;
    least = sums = cost;
    c.g = g;
    c.gz = gz;
    c.mx = mx;
    c.my = my;
  }
  const double direct = 0.8 * 26.0 * nx * ny * natoms;  // as worth() takes them
  c.taken = sums + interpolation_cost(n[0], n[1], nx, ny) < (limit ? *limit : direct);
  return c;
}

}  // namespace

size_t surf_scan_bytes(int nx, int ny, int nmol) { return scan_layout(nx, ny, nmol).total; }

int surf_scan(const SurfInput &in, void *scan, void *digest, hipStream_t s) {
  const ScanLayout l = scan_layout(in.nx, in.ny, in.nmol);
  char *w = (char *)scan;
  const MolInfo one = in.d_mols ? MolInfo{} : in.h_mols[0];
  const ScanArgs sc{in.hkl,
                    in.nx,
                    in.ny,
                    l.list_blocks,
                    in.atoms,
                    in.atom_b,
                    in.d_mols,
                    one,
                    true,
                    (SurfFit *)(w + l.fit),
                    (float *)(w + l.dev),
                    (SurfRecord *)(w + l.records),
                    (double *)(w + l.centres)};
  hipLaunchKernelGGL(surface_scan_kernel, dim3(l.list_blocks + in.nmol * kSurfAtomBlocks), dim3(kT), 0, s, sc);
  const DigestArgs d{sc.fit, sc.records,  l.list_blocks,        in.d_mols,  one,
                     in.segs, in.ff,      in.b_global,          in.atom_b != nullptr, sc.centres,
                     (SurfHead *)digest,  (SurfDigest *)((char *)digest + sizeof(SurfHead))};
  hipLaunchKernelGGL(surface_digest_kernel, dim3(in.nmol), dim3(kT), 0, s, d);
  SPSIM_HIP_TRY(hipGetLastError());
  return SPSIM_HIP_OK;
}

SurfPlan *surf_plan_choose(const SurfInput &in, const void *digest) {
  const SurfHead &head = *(const SurfHead *)digest;
  const SurfDigest *mols = (const SurfDigest *)((const char *)digest + sizeof(SurfHead));
  AxisSlopes along_x(head.slope_x), along_y(head.slope_y);
  SurfPlan *p = new SurfPlan;
  p->in = in;
  p->takes.assign(in.npatterns, 0);
  std::vector<Choice> last(in.nmol);  // of a molecule's last pattern
  std::vector<SurfJob> &jobs = p->jobs;
  for (int i = 0; i < in.npatterns; ++i) {
    const int m = in.pattern_mol ? in.pattern_mol[i] : (in.nmol == 1 ? 0 : i);
    const int natoms = in.h_mols[m].atom_end - in.h_mols[m].atom_begin;
    // rotations differ from 1 by rounding: one node count serves them
    double norm = in.rot9 ? rotation_norm(in.rot9 + 9 * (size_t)i) : 1.0;
    if (std::fabs(norm - 1.0) < 1e-6) norm = 1.0;
    Choice &ch = last[m];
    if (ch.norm != norm) {
      ch = choose(head, along_x, along_y, mols[m].mol, norm, in.nx, in.ny, natoms, in.limit ? in.limit + m : nullptr);
      if (ch.taken) {
        auto find = [](auto &list, auto same) {
          for (size_t k = 0; k < list.size(); ++k)
            if (same(list[k])) return (int)k;
          list.emplace_back();
          return (int)list.size() - 1;
        };
        ch.shape = find(p->shapes, [&](const SurfShape &sh) { return sh.ax.n == ch.ax.n && sh.ay.n == ch.ay.n; });
        p->shapes[ch.shape].ax = ch.ax;
        p->shapes[ch.shape].ay = ch.ay;
        if (ch.g > 0) {
          ch.coarse = find(p->coarse, [&](const SurfCoarse &co) {
            return co.ax.n == ch.mx && co.ay.n == ch.my && co.fx.n == ch.ax.n && co.fy.n == ch.ay.n;
          });
          p->coarse[ch.coarse] = SurfCoarse{axis_of(ch.mx), axis_of(ch.my), ch.ax, ch.ay, nullptr, nullptr, nullptr};
        }
      }
    }
    if (!ch.taken) continue;
    p->takes[i] = 1;
    SurfJob j{};
    j.ok = 1;
    j.nx = in.nx;
    j.ny = in.ny;
    j.sh = p->shapes[ch.shape];
    j.shape = ch.shape;
    j.atoms = in.atoms + in.h_mols[m].atom_begin;
    j.atom_b = in.atom_b ? in.atom_b + in.h_mols[m].atom_begin : nullptr;
    j.segs = in.segs + in.h_mols[m].seg_begin;
    j.nsegs = in.h_mols[m].nseg;
    j.natoms = natoms;
    j.has_rot = in.rot9 != nullptr;
    if (in.rot9) std::copy(in.rot9 + 9 * (size_t)i, in.rot9 + 9 * (size_t)(i + 1), j.rot);
    std::copy(mols[m].centre, mols[m].centre + 3, j.r0);
    std::copy(head.normal, head.normal + 3, j.normal);
    const bool octants = head.sym == 2 && j.sh.ax.n == j.sh.ay.n;
    if (ch.g > 0) {
      SurfCells &c = j.c;
      c.g = ch.g;
      c.gz = ch.gz;
      c.extent = mols[m].mol.radius * norm;
      c.co = p->coarse[ch.coarse];
      j.coarse = ch.coarse;
      cell_tiling(ch.mx, ch.my, octants && ch.mx == ch.my, &c.per_lane, &c.tiles);
      j.per_lane = 1;
      j.tiles = (j.sh.ax.n * j.sh.ay.n + kT - 1) / kT;
    } else {
      // a group has work enough for every tiling: the one of the least work
      node_tiling(j.sh.ax.n, j.sh.ay.n, octants, 1LL << 25, &j.per_lane, &j.tiles);
    }
    j.pattern = i;
    jobs.push_back(j);
  }
  if (jobs.empty()) {
    delete p;
    return nullptr;
  }
  // those with cells first, and largest first, so that a group's patterns need similar grids
  std::stable_sort(jobs.begin(), jobs.end(), [](const SurfJob &a, const SurfJob &b) {
    if ((a.c.g > 0) != (b.c.g > 0)) return a.c.g > 0;
    return (double)a.sh.ax.n * a.sh.ay.n * a.natoms > (double)b.sh.ax.n * b.sh.ay.n * b.natoms;
  });
  const int slots = resident_slots(nodes_kernel(in.atom_b != nullptr, false), in.cus);
  size_t ws_bytes = 0;
  for (int first = 0; first < (int)jobs.size();) {
    SurfPlan::Group g{first, 0, (int)p->items.size(), 0, 0, 0, 0, false, 0, CellBounds{}};
    size_t at = 0;
    while (first + g.count < (int)jobs.size() && g.count < 4096) {
      SurfJob probe = jobs[first + g.count];
      probe.splits = 4;  // a typical group's; only the group's size depends on it
      const size_t end = place(&probe, in.nx, nullptr, at);
      if (g.count > 0 && (end > kGroupBytes || (probe.c.g == 0 && g.celled > 0))) break;
      at = end;
      g.celled += probe.c.g > 0;
      g.max_nodes = std::max(g.max_nodes, probe.sh.ax.n * probe.sh.ay.n);
      g.max_ny = std::max(g.max_ny, probe.sh.ay.n);
      g.max_atoms = std::max(g.max_atoms, probe.natoms);
      ++g.count;
    }
    for (int i = first; i < first + g.celled; ++i) {
      SurfJob &j = jobs[i];
      const SurfCells &c = j.c;
      CellBounds &b = g.cells;
      j.splits = cell_splits(j.sh.ax.n, j.sh.ay.n, g.celled, 1LL << 40);
      const int cells = c.g * c.g * c.gz;
      b.cells = std::max(b.cells, cells);
      b.items = std::max(b.items, (long long)(j.natoms / cell_range(j.natoms) + cells) * c.tiles);
      b.nxn = std::max(b.nxn, j.sh.ax.n);
      b.nyn = std::max(b.nyn, j.sh.ay.n);
      b.splits = std::max(b.splits, j.splits);
    }
    g.cells.items = std::min(g.cells.items, std::max(64LL, 32LL * in.cus / std::max(1, g.celled)));
    g.cells.rows = std::max(64, 8 * in.cus / std::max(1, g.celled));
    split_group(jobs, first, g.count, slots, &p->items);
    g.nitems = (int)p->items.size() - g.item_first;
    at = 0;
    for (int i = first; i < first + g.count; ++i) {
      at = place(&jobs[i], in.nx, nullptr, at);
      g.split = g.split || jobs[i].splits > 1;
    }
    ws_bytes = std::max(ws_bytes, at);
    p->groups.push_back(g);
    first += g.count;
  }
  p->in.h_mols = nullptr;  // the caller's arrays
  p->in.pattern_mol = nullptr;
  p->in.rot9 = nullptr;
  p->in.limit = nullptr;
  p->at_coarse = align_up(sizeof(SurfShape) * p->shapes.size());
  p->at_jobs = p->at_coarse + align_up(sizeof(SurfCoarse) * p->coarse.size());
  p->at_items = p->at_jobs + align_up(sizeof(SurfJob) * jobs.size());
  p->at_tables = p->at_items + align_up(sizeof(SurfItem) * p->items.size());
  size_t at = p->at_tables;
  for (SurfShape &sh : p->shapes) at = place_tables(&sh, in.nx, in.ny, nullptr, at);
  for (SurfCoarse &co : p->coarse) at = place_tables(&co, nullptr, at);
  p->at_ws = at;
  p->bytes = at + ws_bytes;
  return p;
}

size_t surf_plan_bytes(const SurfPlan *p) { return p->bytes; }

int surf_plan_bind(SurfPlan *p, const void *scan, void *mem, hipStream_t s, bool wait) {
  const SurfInput &in = p->in;
  const ScanLayout l = scan_layout(in.nx, in.ny, in.nmol);
  char *w = (char *)mem;
  size_t at = p->at_tables;
  for (SurfShape &sh : p->shapes) at = place_tables(&sh, in.nx, in.ny, w, at);
  for (SurfCoarse &co : p->coarse) at = place_tables(&co, w, at);
  for (const SurfPlan::Group &g : p->groups) {
    at = p->at_ws;
    for (int i = g.first; i < g.first + g.count; ++i) {
      p->jobs[i].sh = p->shapes[p->jobs[i].shape];
      if (p->jobs[i].c.g > 0) p->jobs[i].c.co = p->coarse[p->jobs[i].coarse];
      at = place(&p->jobs[i], in.nx, w, at);
    }
  }
  std::vector<char> &image = p->image;
  image.resize(p->at_tables);
  std::copy(p->shapes.begin(), p->shapes.end(), (SurfShape *)image.data());
  std::copy(p->coarse.begin(), p->coarse.end(), (SurfCoarse *)(image.data() + p->at_coarse));
  std::copy(p->jobs.begin(), p->jobs.end(), (SurfJob *)(image.data() + p->at_jobs));
  std::copy(p->items.begin(), p->items.end(), (SurfItem *)(image.data() + p->at_items));
  SPSIM_HIP_TRY(hipMemcpyAsync(w, image.data(), image.size(), hipMemcpyHostToDevice, s));
  const int nshapes = (int)p->shapes.size();
  for (int first = 0; first < nshapes; first += 4096)
    hipLaunchKernelGGL(surface_tables_kernel, dim3(256, 2, std::min(4096, nshapes - first)), dim3(kT), 0, s,
                       (const SurfFit *)((const char *)scan + l.fit), (const SurfShape *)w + first, in.nx, in.ny);
  const int ncoarse = (int)p->coarse.size();
  for (int first = 0; first < ncoarse; first += 4096)
    hipLaunchKernelGGL(surface_coarse_kernel, dim3(64, 2, std::min(4096, ncoarse - first)), dim3(kT), 0, s,
                       (const SurfFit *)((const char *)scan + l.fit), (const SurfCoarse *)(w + p->at_coarse) + first);
  SPSIM_HIP_TRY(hipGetLastError());
  if (wait) {  // the copy reads image
    SPSIM_HIP_TRY(hipStreamSynchronize(s));
    image = std::vector<char>();
  }
  p->dev = (const float *)((const char *)scan + l.dev);
  p->d_jobs = (const SurfJob *)(w + p->at_jobs);
  p->d_items = (const SurfItem *)(w + p->at_items);
  return SPSIM_HIP_OK;
}

int surf_plan_create(const SurfInput &in, SurfPlan **out) {
  *out = nullptr;
  if (in.nx < kSurfMinSide || in.ny < kSurfMinSide) return SPSIM_HIP_OK;
  const size_t scan_bytes = surf_scan_bytes(in.nx, in.ny, in.nmol), digest_bytes = surf_digest_bytes(in.nmol);
  auto alloc = [](void **m, size_t bytes) {
    const hipError_t e = hipMalloc(m, bytes);
    if (e == hipSuccess) return SPSIM_HIP_OK;
    (void)hipGetLastError();  // the caller may go on without the plan
    return fail(SPSIM_HIP_ERR_NOMEM, "hipMalloc(%zu) failed: %s", bytes, hipGetErrorString(e));
  };
  void *scan = nullptr, *mem = nullptr;
  SPSIM_TRY(alloc(&scan, scan_bytes + digest_bytes));
  void *digest = (char *)scan + scan_bytes;
  std::vector<char> h(digest_bytes);
  int rc = surf_scan(in, scan, digest, nullptr);
  if (rc == SPSIM_HIP_OK) {
    const hipError_t e = hipMemcpy(h.data(), digest, digest_bytes, hipMemcpyDeviceToHost);
    if (e != hipSuccess) rc = hip_fail(e, "surface scan");
  }
  SurfPlan *p = rc == SPSIM_HIP_OK ? surf_plan_choose(in, h.data()) : nullptr;
  if (!p) {
    (void)hipFree(scan);
    return rc;
  }
  p->owned.push_back(scan);
  rc = alloc(&mem, p->bytes);
  if (rc == SPSIM_HIP_OK) {
    p->owned.push_back(mem);
    rc = surf_plan_bind(p, scan, mem, nullptr, true);
  }
  if (rc != SPSIM_HIP_OK) {
    surf_plan_destroy(p);
    return rc;
  }
  *out = p;
  return SPSIM_HIP_OK;
}

bool surf_plan_takes(const SurfPlan *p, int pattern) { return p && p->takes[pattern]; }

int surf_plan_run(const SurfPlan *p, float2 *F, float *I, hipStream_t s) {
  const SurfInput &in = p->in;
  const bool has_b = in.atom_b != nullptr;
  const int slots = resident_slots(nodes_kernel(has_b, false), in.cus);
  for (const SurfPlan::Group &g : p->groups) {
    const int wgs = std::max(16, std::min((g.max_atoms + kT - 1) / kT, 4 * in.cus / g.count));
    hipLaunchKernelGGL(surface_prepare_kernel, dim3(wgs, g.count), dim3(kT), 0, s, p->d_jobs, g.first, has_b);
    const SurfItem *items = p->d_items + g.item_first;
    const int blocks = std::min(g.nitems, slots);
    if (g.nitems > 0) SPSIM_TRY(launch_nodes(p->d_jobs, items, g.nitems, blocks, in.ff, in.b_global, has_b, nullptr, s));
    if (g.celled > 0) launch_cells(p->d_jobs, g.first, g.celled, g.cells, in.ff, in.b_global, has_b, s);
    launch_interpolation(p->d_jobs, g.first, g.count, in.nx, in.ny, g.split ? g.max_nodes : 0, g.max_ny, p->dev, in.hkl,
                         F, I, s);
  }
  SPSIM_HIP_TRY(hipGetLastError());
  return SPSIM_HIP_OK;
}

void surf_plan_destroy(SurfPlan *p) {
  if (!p) return;
  for (void *m : p->owned) (void)hipFree(m);
  delete p;
}

}  // namespace spsim
