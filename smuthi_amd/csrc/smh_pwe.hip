// Plane wave expansion near field on the GPU: E (or omega H) of
//   F(r) = int kappa dkappa int dalpha f(kappa, alpha) e^{i (kx x + ky y + kz z)}
// by the nested trapezoid rule (alpha inner, kappa outer) of
// PlaneWaveExpansion.electric_field / magnetic_field (fields/expansions.py:635-782).
//
// Layout. Points are ordered into leaves of at most kLeaf points by recursive
// median splits, in-plane first: a leaf is narrow in x and y and may be tall in
// z. The leaf origin r0 splits every phase as e^{i k.r0} e^{i k.(r - r0)}: the
// first factor is folded into the (kappa, alpha) coefficients once per leaf in
// FP64. Workgroups take a leaf and a range of kappa; a last kernel adds the
// ranges' sums in FP64 and puts the points back in the caller's order.
//
// The sum over alpha, chosen per leaf by its in-plane radius R:
// * pwe_harmonics_kernel where kappa R is small against the number of azimuths:
//   e^{i kappa rho cos(alpha - phi)} = J_0 + 2 sum_m i^m J_m(kappa rho) cos(m (alpha - phi))
//   (Jacobi-Anger), so the leaf's coefficients become a few harmonics per kappa,
//   shared by all its points: M ~ kappa R + 10 terms per point instead of n_alpha.
//   Points above one another need order 0 only (pwe_column_kernel).
// * pwe_field_kernel otherwise: one thread per point, one term per alpha. The
//   per-term phase k.(r - r0) is small and FP32 keeps it accurate; per term the
//   FP32 kernel spends one native sin and cos (argument in revolutions) and, on
//   the complex part of the contour only, one exp2, plus three complex
//   multiply-adds.
#include <algorithm>
#include <cmath>
#include <complex>
#include <cstring>
#include <numeric>
#include <vector>

#include "smh_common.h"
#include "smh_radial_kernel.h"

namespace {

constexpr int kLeaf = 256;
constexpr double kTwoPi = 6.283185307179586476925286766559;
constexpr double kLog2e = 1.4426950408889634073599246810019;

struct PweArgs {
  const double2* F;    // [3][n_k][n_a] weighted integrand coefficients
  const double2* kp;   // [n_k]
  const double2* kz;   // [n_k]
  const double* ca;    // cos alpha [n_a]
  const double* sa;    // sin alpha [n_a]
  const void* trig;    // [n_a, padded][2][kMaxM + 1] cos, sin(m alpha) of Real (harmonics)
  const double* pts;   // [n_pts][3], leaf order
  const int* leaf;     // [n_leaves + 1] offsets into pts
  const double* org;   // [n_leaves][4] leaf origins and in-plane radii
  const int* list;     // the launch's leaves
  double2* part;       // [splits][3][n_pts], leaf order
  int64_t n_pts;
  int n_k, n_a, kc;    // kc: kappa per LDS chunk (pwe_field_kernel)
  int per_split;       // kappa per blockIdx.y
};

template <typename Real>
struct PweMath;

template <>
struct PweMath<float> {
  // e^{i 2 pi t} for |t| of a few revolutions (native v_sin / v_cos)
  static __device__ inline void cis_rev(float t, float& c, float& s) {
    s = __builtin_amdgcn_sinf(t);
    c = __builtin_amdgcn_cosf(t);
  }
  static __device__ inline float exp2_(float x) { return __builtin_amdgcn_exp2f(x); }
};

template <>
struct PweMath<double> {
  static __device__ inline void cis_rev(double t, double& c, double& s) { sincos(kTwoPi * t, &s, &c); }
  static __device__ inline double exp2_(double x) { return exp2(x); }
};

// A wavenumber in turns (over 2 pi) per length, to twice FP64's digits, and the
// fraction of a turn of k s: the product less its whole turns is rounded once,
// at the size of the fraction (a rounded product would leave FP64 phases 1e-16
// of the whole argument, some hundred radians over an array).
struct Turns {
  double hi, lo;
};
__device__ inline Turns turns_of(double k) {
  constexpr double kInvHi = 0.15915494309189535, kInvLo = -9.839338337591243e-18;  // 1 / (2 pi)
  const double hi = k * kInvHi;
  return {hi, fma(k, kInvLo, fma(k, kInvHi, -hi))};
}
__device__ inline double turn_fraction(Turns k, double s) {
  return fma(k.lo, s, fma(k.hi, s, -rint(k.hi * s)));
}

// e^{i 2 pi t} of a fraction of a turn
__device__ inline void cis_turns(double t, double& c, double& s) { sincospi(2.0 * t, &s, &c); }
__device__ inline void cis_turns(double t, float& c, float& s) { PweMath<float>::cis_rev((float)t, c, s); }

// e^{i kz dz}, the argument reduced in FP64 (leaves may be tall)
template <typename Real>
__device__ inline void z_phase(double2 kz, double dz, Real& c, Real& s) {
  cis_turns(turn_fraction(turns_of(kz.x), dz), c, s);
  if (kz.y != 0.0) {
    const Real m = PweMath<Real>::exp2_((Real)(-kz.y * kLog2e * dz));
    c *= m;
    s *= m;
  }
}

// Integrand coefficients F(c, k, alpha) with the quadrature weights
// (expansions.py:676-699 for E, :745-766 for H); wk includes the kappa factor.
__global__ void pwe_coefficients_kernel(int kind, int n_k, int n_a, const double2* __restrict__ g,
                                        const double2* __restrict__ kp, const double2* __restrict__ kz,
                                        const double* __restrict__ ca, const double* __restrict__ sa,
                                        const double2* __restrict__ wk, const double* __restrict__ wa, double2 kk,
                                        double2* F) {
  const int64_t n = (int64_t)n_k * n_a, i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int k = (int)(i / n_a), j = (int)(i - (int64_t)k * n_a);
  using C = cplx<double>;
  auto ld = [](double2 v) { return C{v.x, v.y}; };
  const C g0 = ld(g[i]), g1 = ld(g[n + i]), kpk = ld(kp[k]), kzk = ld(kz[k]), q = ld(kk);
  const double c = ca[j], s = sa[j];
  C fx, fy, fz;
  if (kind == 0) {
    const C t = cmul(cdiv(kzk, q), g1);
    fx = cadd(cscale(g0, -s), cscale(t, c));
    fy = cadd(cscale(g0, c), cscale(t, s));
    fz = cscale(cmul(cdiv(kpk, q), g1), -1.0);
  } else {
    const C t = cmul(kzk, g0), u = cmul(q, g1);
    fx = cscale(cadd(cscale(t, c), cscale(u, s)), -1.0);
    fy = cadd(cscale(t, -s), cscale(u, c));
    fz = cmul(kpk, g0);
  }
  const C w = cscale(ld(wk[k]), wa[j]);
  const C f[3] = {cmul(w, fx), cmul(w, fy), cmul(w, fz)};
#pragma unroll
  for (int d = 0; d < 3; ++d) F[d * n + i] = make_double2(f[d].re, f[d].im);
}

// Largest |z| whose expansion may end at order M: the sum of 2 |J_m(z)| over
// m > M stays below 1e-9 (FP32) and 1e-16 (FP64).
constexpr int kMaxM = 63;
#define SMH_ORDER_LIMIT_32 \
    9.9e-10, 6.3e-05, 0.00288, 0.0209, 0.0717, 0.168, 0.316, 0.516, 0.765, 1.06, 1.4, 1.77, 2.18, 2.62, 3.09, 3.58, \
    4.1, 4.63, 5.19, 5.76, 6.35, 6.95, 7.56, 8.19, 8.83, 9.48, 10.1, 10.8, 11.5, 12.2, 12.9, 13.6, \
    14.3, 15, 15.7, 16.5, 17.2, 17.9, 18.7, 19.4, 20.2, 20.9, 21.7, 22.5, 23.3, 24, 24.8, 25.6, \
    26.4, 27.2, 28, 28.8, 29.6, 30.4, 31.2, 32, 32.8, 33.6, 34.4, 35.2, 36, 36.9, 37.7, 38.5
#define SMH_ORDER_LIMIT_64 \
    6.9e-17, 2e-08, 1.34e-05, 0.000372, 0.00286, 0.0115, 0.0317, 0.0689, 0.128, 0.212, 0.323, 0.462, 0.63, 0.826, 1.05, 1.3, \
    1.58, 1.88, 2.2, 2.54, 2.91, 3.29, 3.69, 4.11, 4.55, 5, 5.47, 5.95, 6.44, 6.95, 7.47, 8, \
    8.54, 9.09, 9.65, 10.2, 10.8, 11.4, 12, 12.6, 13.2, 13.8, 14.4, 15.1, 15.7, 16.3, 17, 17.6, \
    18.3, 19, 19.6, 20.3, 21, 21.7, 22.4, 23.1, 23.8, 24.5, 25.2, 25.9, 26.6, 27.3, 28, 28.7
__constant__ double kOrderLimit32[kMaxM + 1] = {SMH_ORDER_LIMIT_32};
__constant__ double kOrderLimit64[kMaxM + 1] = {SMH_ORDER_LIMIT_64};
__host__ __device__ inline int order_for(const double* limit, double z) {
  int m = 0;
  for (int step = 32; step > 0; step >>= 1)
    if (m + step <= kMaxM && z > limit[m + step - 1]) m += step;
  return m;  // kMaxM where z is beyond the table
}

// 2^e; FP32: the whole part of e goes into the exponent field, so that e may be large (rounded to FP32 as a
// whole it would cost 6e-8 |e| of the result)
__device__ inline double exp2_split(double e, double) { return exp2(e); }
__device__ inline float exp2_split(double e, float) {
  const double w = rint(fmax(-1e4, fmin(1e4, e)));
  return ldexpf(PweMath<float>::exp2_((float)(e - w)), (int)w);
}

// Host: the order a leaf with largest |kappa| R = z needs, -1 beyond kMaxM.
int max_order(int precision, double z) {
  static const double limit32[kMaxM + 1] = {SMH_ORDER_LIMIT_32}, limit64[kMaxM + 1] = {SMH_ORDER_LIMIT_64};
  const double* limit = precision == SMH_FP32 ? limit32 : limit64;
  return z > limit[kMaxM] ? -1 : order_for(limit, z);
}

// cos, sin(m alpha) in the order of the MFMA's rows, zero beyond n_a
template <typename Real>
__global__ void pwe_trig_kernel(int n_a, int rows, const double* __restrict__ alpha, Real* trig) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= rows * (kMaxM + 1)) return;
  const int j = i / (kMaxM + 1), m = i - j * (kMaxM + 1);
  double s = 0.0, c = 0.0;
  if (j < n_a) sincos(m * alpha[j], &s, &c);
  trig[(size_t)j * 2 * (kMaxM + 1) + m] = (Real)c;
  trig[(size_t)j * 2 * (kMaxM + 1) + kMaxM + 1 + m] = (Real)s;
}

// Field of a leaf of points above one another: per kappa one sum over alpha,
// A = sum F e^{i kp (x0 cos + y0 sin)}, serves all its points. A wave takes a
// kappa at a time, its lanes the azimuths, then the points (four a lane). Bound
// by one FP64 sincos per (leaf, kappa, azimuth) and the z phases. 65,536 points
// of a vertical cut, 1042 x 180 waves, FP32: 18.2 ms with one term per azimuth
// and point, 2.3 ms through pwe_harmonics_kernel, 0.45 ms in this form, which
// needs no LDS and no barriers per kappa.
template <typename Real>
__global__ void __launch_bounds__(256) pwe_column_kernel(PweArgs a) {
  constexpr int PT = kLeaf / 64;
  __shared__ double tot[kLeaf][6];
  const int leaf = a.list[blockIdx.x], tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int p0 = a.leaf[leaf], p1 = a.leaf[leaf + 1], nu = (p1 - p0 + 63) / 64;
  const double x0 = a.org[4 * leaf], y0 = a.org[4 * leaf + 1], z0 = a.org[4 * leaf + 2];
  double dz[PT], acc[PT][6];
#pragma unroll
  for (int u = 0; u < PT; ++u) {
    dz[u] = a.pts[3 * min(p0 + lane + 64 * u, p1 - 1) + 2] - z0;  // (lanes beyond the leaf are not stored)
#pragma unroll
    for (int c = 0; c < 6; ++c) acc[u][c] = 0.0;
  }
  const int k_end = min(a.n_k, ((int)blockIdx.y + 1) * a.per_split);
  for (int k = (int)blockIdx.y * a.per_split + wave; k < k_end; k += 4) {
    const double2 kp = a.kp[k], kz = a.kz[k];
    const Turns kturn = turns_of(kp.x);
    double A[6] = {0, 0, 0, 0, 0, 0};
    for (int j = lane; j < a.n_a; j += 64) {
      const double sxy = x0 * a.ca[j] + y0 * a.sa[j];
      double er, ei;
      cis_turns(turn_fraction(kturn, sxy), er, ei);
      if (kp.y != 0.0) {
        const double mag = exp(-kp.y * sxy);
        er *= mag;
        ei *= mag;
      }
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const double2 v = a.F[((size_t)c * a.n_k + k) * a.n_a + j];
        A[2 * c] += v.x * er - v.y * ei;
        A[2 * c + 1] += v.x * ei + v.y * er;
      }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
#pragma unroll
      for (int c = 0; c < 6; ++c) A[c] += __shfl_xor(A[c], off);
    double er, ei;  // e^{i kz z0}
    z_phase(kz, z0, er, ei);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const double t = A[2 * d] * er - A[2 * d + 1] * ei;
      A[2 * d + 1] = A[2 * d] * ei + A[2 * d + 1] * er;
      A[2 * d] = t;
    }
#pragma unroll
    for (int u = 0; u < PT; ++u) {
      if (u >= nu) break;
      Real zc, zs;
      z_phase(kz, dz[u], zc, zs);
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        acc[u][2 * d] += A[2 * d] * zc - A[2 * d + 1] * zs;
        acc[u][2 * d + 1] += A[2 * d] * zs + A[2 * d + 1] * zc;
      }
    }
  }
  // the waves' sums, one wave after the other
  for (int w = 0; w < 4; ++w) {
    if (wave == w)
#pragma unroll
      for (int u = 0; u < PT; ++u)
#pragma unroll
        for (int c = 0; c < 6; ++c) {
          double* t = &tot[lane + 64 * u][c];
          *t = w ? *t + acc[u][c] : acc[u][c];
        }
    __syncthreads();
  }
  if (p0 + tid < p1) {
    double2* part = a.part + (size_t)3 * blockIdx.y * a.n_pts + p0 + tid;
#pragma unroll
    for (int c = 0; c < 3; ++c) part[c * a.n_pts] = make_double2(tot[tid][2 * c], tot[tid][2 * c + 1]);
  }
}

// Field of one leaf over a range of kappa through azimuthal harmonics, KC kappa
// at a time: (1) the leaf coefficients f(kappa, alpha) in FP64 phases, kAC
// azimuths at a time in LDS; (2) the harmonics A_m = sum_alpha f cos(m alpha),
// B_m = sum f sin(m alpha) as a product on the MFMA (rows (cos | sin, m), columns
// (kappa, component, re | im), the sum over alpha), times 2 i^m into LDS; (3) per
// wave one kappa at a time and per lane four points: sum_m J_m(kappa rho)
// (A_m cos(m phi) + B_m sin(m phi)) with J_m from Miller's backward recurrence,
// in FP64 throughout (its range holds the unnormalised values; FP64 and unpacked
// FP32 issue at one rate on this chip). Bound by the VALU of (3): 20
// instructions per order and point, against 26 and four transcendental ones per
// azimuth and point in pwe_field_kernel; (2) costs about a third of it at M = 15.
constexpr int kAC = 192;
template <typename Real, int KC>
__global__ void __launch_bounds__(256) pwe_harmonics_kernel(PweArgs a) {
  using M = smh::Mfma<Real>;
  constexpr int MR = 256 / KC;                 // orders held: 32 or 64
  constexpr int CT = (KC * 6 + 15) / 16;       // column tiles
  constexpr int UW = 2 * (MR / 16) * CT / 4;   // result tiles per wave at most
  constexpr int PT = kLeaf / 64;               // points per lane
  __shared__ __align__(16) unsigned char smem[KC * kAC * 6 * sizeof(Real) + KC * MR * 12 * sizeof(double)];
  Real* f = reinterpret_cast<Real*>(smem);                                              // [KC][kAC][6]
  double* G = reinterpret_cast<double*>(smem + KC * kAC * 6 * sizeof(Real));            // [KC][MR][A 6 | B 6]
  static_assert(sizeof(smem) >= kLeaf * 6 * sizeof(double), "the waves' sums are added in the staging space");
  const double* limit = sizeof(Real) == 4 ? kOrderLimit32 : kOrderLimit64;
  const int leaf = a.list[blockIdx.x], tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, q = lane >> 4, r = lane & 15;
  const int p0 = a.leaf[leaf], p1 = a.leaf[leaf + 1];
  const double x0 = a.org[4 * leaf], y0 = a.org[4 * leaf + 1], z0 = a.org[4 * leaf + 2], radius = a.org[4 * leaf + 3];
  double irho[PT], cp[PT], sp[PT], dz[PT];  // 1 / rho, cos phi, sin phi, z - z0 of the lane's points
  double ec[PT], es[PT];                    // e^{i m_at phi}
  double acc[PT][6];
#pragma unroll
  for (int u = 0; u < PT; ++u) {
    const int p = min(p0 + lane + 64 * u, p1 - 1);  // (lanes beyond the leaf repeat its last point, not stored)
    const double dx = a.pts[3 * p] - x0, dy = a.pts[3 * p + 1] - y0;
    const double rho = sqrt(dx * dx + dy * dy);
    irho[u] = 1.0 / fmax(rho, 1e-20);
    cp[u] = rho > 0 ? dx / rho : 1.0;
    sp[u] = rho > 0 ? dy / rho : 0.0;
    dz[u] = a.pts[3 * p + 2] - z0;
    ec[u] = 1.0;
    es[u] = 0.0;
#pragma unroll
    for (int c = 0; c < 6; ++c) acc[u][c] = 0.0;
  }
  int m_at = 0;

  // one kappa's harmonics at the lane's points (J_m complex on the lossy part of the contour)
  auto sum_points = [&](auto lossy, const double* Gk, double2 kp, double2 kz, int mc) {
    constexpr bool L = decltype(lossy)::value;
    // e^{i mc phi} follows the order from one kappa to the next
    for (; m_at < mc; ++m_at)
#pragma unroll
      for (int u = 0; u < PT; ++u) {
        const double c = ec[u] * cp[u] - es[u] * sp[u];
        es[u] = ec[u] * sp[u] + es[u] * cp[u];
        ec[u] = c;
      }
    for (; m_at > mc; --m_at)
#pragma unroll
      for (int u = 0; u < PT; ++u) {
        const double c = ec[u] * cp[u] + es[u] * sp[u];
        es[u] = es[u] * cp[u] - ec[u] * sp[u];
        ec[u] = c;
      }
    double in[PT][6], jr[PT], ji[PT], lr[PT], li[PT], nr[PT], ni[PT], c_[PT], s_[PT], tr[PT], ti[PT];
    const double k2 = kp.x * kp.x + kp.y * kp.y;
#pragma unroll
    for (int u = 0; u < PT; ++u) {
#pragma unroll
      for (int c = 0; c < 6; ++c) in[u][c] = 0.0;
      jr[u] = mc > 0 ? 1e-280 : 1.0;  // order mc + 2, the one above it zero; M = 0: J_0 = 1
      ji[u] = lr[u] = li[u] = nr[u] = ni[u] = 0.0;
      c_[u] = ec[u];
      s_[u] = es[u];
      tr[u] = k2 > 0 ? 2.0 * kp.x / k2 * irho[u] : 0.0;  // 2 / (kappa rho)
      ti[u] = L ? -2.0 * kp.y / k2 * irho[u] : 0.0;
    }
    // (J_m, J_m+1) -> (J_m-1, J_m)
    auto down = [&](int u, int m) {
      const double ar = m * tr[u];
      if constexpr (L) {
        const double ai = m * ti[u];
        const double xr = fma(ar, jr[u], fma(-ai, ji[u], -lr[u])), xi = fma(ar, ji[u], fma(ai, jr[u], -li[u]));
        lr[u] = jr[u];
        li[u] = ji[u];
        jr[u] = xr;
        ji[u] = xi;
      } else {
        const double x = fma(ar, jr[u], -lr[u]);
        lr[u] = jr[u];
        jr[u] = x;
      }
    };
    auto add_order = [&](int m) {
      const double2* g = reinterpret_cast<const double2*>(Gk + 12 * m);
      double2 A[3], B[3];
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        A[d] = g[d];
        B[d] = g[3 + d];
      }
#pragma unroll
      for (int u = 0; u < PT; ++u) {
        const double vr = jr[u] * c_[u], wr = jr[u] * s_[u];
        if constexpr (L) {
          const double vi = ji[u] * c_[u], wi = ji[u] * s_[u];
#pragma unroll
          for (int d = 0; d < 3; ++d) {
            in[u][2 * d] = fma(vr, A[d].x, fma(-vi, A[d].y, fma(wr, B[d].x, fma(-wi, B[d].y, in[u][2 * d]))));
            in[u][2 * d + 1] = fma(vr, A[d].y, fma(vi, A[d].x, fma(wr, B[d].y, fma(wi, B[d].x, in[u][2 * d + 1]))));
          }
        } else {
#pragma unroll
          for (int d = 0; d < 3; ++d) {
            in[u][2 * d] = fma(vr, A[d].x, fma(wr, B[d].x, in[u][2 * d]));
            in[u][2 * d + 1] = fma(vr, A[d].y, fma(wr, B[d].y, in[u][2 * d + 1]));
          }
        }
        if (!(m & 1)) {  // J_0 + 2 sum J_2k = 1
          const double e = m ? 2.0 : 1.0;
          nr[u] = fma(e, jr[u], nr[u]);
          if (L) ni[u] = fma(e, ji[u], ni[u]);
        }
      }
    };
    if (mc > 0) {
#pragma unroll
      for (int u = 0; u < PT; ++u) {
        down(u, mc + 2);
        down(u, mc + 1);
      }
    }
    for (int m = mc; m > 0; --m) {
      add_order(m);
#pragma unroll
      for (int u = 0; u < PT; ++u) {
        down(u, m);
        const double c = c_[u] * cp[u] + s_[u] * sp[u];
        s_[u] = s_[u] * cp[u] - c_[u] * sp[u];
        c_[u] = c;
        // near the axis the values grow by up to 1e24 per order: rescale every fourth one
        if ((m & 3) == 0 && fmax(fabs(jr[u]), L ? fabs(ji[u]) : 0.0) > 1e150) {
          const double down_ = 1e-150;
          jr[u] *= down_;
          lr[u] *= down_;
          nr[u] *= down_;
          if (L) {
            ji[u] *= down_;
            li[u] *= down_;
            ni[u] *= down_;
          }
#pragma unroll
          for (int c2 = 0; c2 < 6; ++c2) in[u][c2] *= down_;
        }
      }
    }
    add_order(0);
#pragma unroll
    for (int u = 0; u < PT; ++u) {
      Real zc, zs;
      z_phase(kz, dz[u], zc, zs);
      // e^{i kz dz} / norm
      double er, ei;
      if constexpr (L) {
        // (the norm's square would leave the range)
        const double w = 1.0 / fmax(fabs(nr[u]), fabs(ni[u])), x = nr[u] * w, y = ni[u] * w;
        const double in2 = w / (x * x + y * y);
        er = ((double)zc * x + (double)zs * y) * in2;
        ei = ((double)zs * x - (double)zc * y) * in2;
      } else {
        const double in1 = 1.0 / nr[u];
        er = (double)zc * in1;
        ei = (double)zs * in1;
      }
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        acc[u][2 * d] += in[u][2 * d] * er - in[u][2 * d + 1] * ei;
        acc[u][2 * d + 1] += in[u][2 * d] * ei + in[u][2 * d + 1] * er;
      }
    }
  };

  const int k_end = min(a.n_k, ((int)blockIdx.y + 1) * a.per_split);
  const Real* trig = reinterpret_cast<const Real*>(a.trig);
  for (int k0 = (int)blockIdx.y * a.per_split; k0 < k_end; k0 += KC) {
    const int kn = min(KC, k_end - k0);
    int mmax = 0;
    for (int kk = 0; kk < kn; ++kk) {
      const double2 kp = a.kp[k0 + kk];
      mmax = max(mmax, order_for(limit, sqrt(kp.x * kp.x + kp.y * kp.y) * radius));
    }
    mmax = min(mmax, MR - 1);  // (the host put the leaf where its orders fit; rounding aside)
    const int mt = (mmax + 16) / 16, units = 2 * mt * CT;  // tiles of 16 orders
    typename M::v4 h[UW];
#pragma unroll
    for (int i = 0; i < UW; ++i) h[i] = typename M::v4{0, 0, 0, 0};
    for (int a0 = 0; a0 < a.n_a; a0 += kAC) {
      const int an = min(kAC, a.n_a - a0), an4 = (an + 3) / 4 * 4;
      __syncthreads();
      // (1) f = F e^{i (kp (x0 cos + y0 sin) + kz z0)}, zero for the azimuths that fill up a step of four and
      // the kappa beyond the range
      for (int j = tid; j < KC * an4; j += blockDim.x) {
        const int kk = j / an4, ia = j - kk * an4;
        Real* dst = f + ((size_t)kk * kAC + ia) * 6;
        if (kk >= kn || ia >= an) {
#pragma unroll
          for (int c = 0; c < 6; ++c) dst[c] = Real(0);
          continue;
        }
        const int k = k0 + kk;
        const double2 kp = a.kp[k], kz = a.kz[k];
        const double sxy = x0 * a.ca[a0 + ia] + y0 * a.sa[a0 + ia];
        double er, ei;
        cis_turns(turn_fraction(turns_of(kp.x), sxy) + turn_fraction(turns_of(kz.x), z0), er, ei);
        if (kp.y != 0.0 || kz.y != 0.0) {
          const double mag = exp(-(kp.y * sxy + kz.y * z0));
          er *= mag;
          ei *= mag;
        }
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          const double2 v = a.F[((size_t)c * a.n_k + k) * a.n_a + a0 + ia];
          dst[2 * c] = (Real)(v.x * er - v.y * ei);
          dst[2 * c + 1] = (Real)(v.x * ei + v.y * er);
        }
      }
      __syncthreads();
      // (2)
#pragma unroll
      for (int i = 0; i < UW; ++i) {
        const int unit = wave + 4 * i;
        if (unit < units) {
          const int ct = unit % CT, row = unit / CT, cs = row / mt, tile = row - cs * mt;
          const int col = min(16 * ct + r, KC * 6 - 1), kk = col / 6, c = col - 6 * kk;
          const Real* A = trig + (size_t)(a0 + q) * 2 * (kMaxM + 1) + cs * (kMaxM + 1) + 16 * tile + r;
          const Real* B = f + ((size_t)kk * kAC + q) * 6 + c;
#pragma unroll 4
          for (int s = 0; s < an4 / 4; ++s) h[i] = M::op(A[(size_t)s * 8 * (kMaxM + 1)], B[24 * s], h[i]);
        }
      }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < UW; ++i) {
      const int unit = wave + 4 * i;
      if (unit < units) {
        const int ct = unit % CT, row = unit / CT, cs = row / mt, tile = row - cs * mt;
        const int col = 16 * ct + r, kk = col / 6, c = col - 6 * kk;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int m = 16 * tile + (M::kRowIs4q ? 4 * q + v : 4 * v + q);
          // times 2 i^m (1 for m = 0): odd orders exchange re and im
          const bool neg = ((m >> 1) ^ (m & c)) & 1;
          const double w = (m ? 2.0 : 1.0) * (double)h[i][v];
          if (col < KC * 6) G[((size_t)kk * MR + m) * 12 + 6 * cs + (c ^ (m & 1))] = neg ? -w : w;
        }
      }
    }
    __syncthreads();
    // (3)
    for (int kk = wave; kk < kn; kk += 4) {
      const double2 kp = a.kp[k0 + kk], kz = a.kz[k0 + kk];
      const int mc = min(MR - 1, order_for(limit, sqrt(kp.x * kp.x + kp.y * kp.y) * radius));
      const double* Gk = G + (size_t)kk * MR * 12;
      if (kp.y != 0.0)
        sum_points(std::true_type{}, Gk, kp, kz, mc);
      else
        sum_points(std::false_type{}, Gk, kp, kz, mc);
    }
  }
  // the waves' sums, one wave after the other
  double* tot = reinterpret_cast<double*>(smem);  // [kLeaf][6]
  for (int w = 0; w < 4; ++w) {
    __syncthreads();
    if (wave == w)
#pragma unroll
      for (int u = 0; u < PT; ++u)
#pragma unroll
        for (int c = 0; c < 6; ++c) {
          double* t = tot + (lane + 64 * u) * 6 + c;
          *t = w ? *t + acc[u][c] : acc[u][c];
        }
  }
  __syncthreads();
  if (p0 + tid < p1) {
    double2* part = a.part + (size_t)3 * blockIdx.y * a.n_pts + p0 + tid;
#pragma unroll
    for (int c = 0; c < 3; ++c) part[c * a.n_pts] = make_double2(tot[tid * 6 + 2 * c], tot[tid * 6 + 2 * c + 1]);
  }
}

template <typename Real>
__global__ void __launch_bounds__(kLeaf) pwe_field_kernel(PweArgs a) {
  using M = PweMath<Real>;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  Real* cs = reinterpret_cast<Real*>(smem_raw);  // [n_a][2] cos, sin
  Real* fl = cs + 2 * a.n_a;                      // [kc][n_a][6] leaf coefficients (re, im) x 3
  const int leaf = a.list[blockIdx.x], tid = threadIdx.x;
  const int p0 = a.leaf[leaf], p1 = a.leaf[leaf + 1];
  const int p = p0 + tid;
  const bool active = p < p1;
  const double x0 = a.org[4 * leaf], y0 = a.org[4 * leaf + 1], z0 = a.org[4 * leaf + 2];
  Real dx = 0, dy = 0;
  double dz = 0;
  if (active) {
    dx = (Real)(a.pts[3 * p] - x0);
    dy = (Real)(a.pts[3 * p + 1] - y0);
    dz = a.pts[3 * p + 2] - z0;
  }
  for (int j = tid; j < a.n_a; j += blockDim.x) {
    cs[2 * j] = (Real)a.ca[j];
    cs[2 * j + 1] = (Real)a.sa[j];
  }
  double acc[6] = {0, 0, 0, 0, 0, 0};
  const int k_end = min(a.n_k, ((int)blockIdx.y + 1) * a.per_split);
  for (int k0 = (int)blockIdx.y * a.per_split; k0 < k_end; k0 += a.kc) {
    const int kn = min(a.kc, k_end - k0);
    __syncthreads();
    // leaf coefficients: F(c, k, alpha) e^{i (kp (x0 cos + y0 sin) + kz z0)} in FP64
    for (int j = tid; j < kn * a.n_a; j += blockDim.x) {
      const int kk = j / a.n_a, ia = j - kk * a.n_a, k = k0 + kk;
      const double2 kp = a.kp[k], kz = a.kz[k];
      const double sxy = x0 * a.ca[ia] + y0 * a.sa[ia];
      // i (kp sxy + kz z0)
      const double ph_re = -(kp.y * sxy + kz.y * z0), ph_im = kp.x * sxy + kz.x * z0;
      double sn, cn;
      sincos(ph_im, &sn, &cn);
      const double mag = exp(ph_re);
      const double er = mag * cn, ei = mag * sn;
      Real* dst = fl + (size_t)j * 6;
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const double2 f = a.F[((size_t)c * a.n_k + k) * a.n_a + ia];
        dst[2 * c] = (Real)(f.x * er - f.y * ei);
        dst[2 * c + 1] = (Real)(f.x * ei + f.y * er);
      }
    }
    __syncthreads();
    for (int kk = 0; kk < kn; ++kk) {
      const double2 kpd = a.kp[k0 + kk], kzd = a.kz[k0 + kk];
      const Real kr = (Real)(kpd.x / kTwoPi);     // revolutions per nm
      const Real ki = (Real)(-kpd.y * kLog2e);    // log2 of the decay per nm
      const bool lossy = kpd.y != 0.0;
      Real in[6] = {0, 0, 0, 0, 0, 0};
      const Real* f = fl + (size_t)kk * a.n_a * 6;
      for (int ia = 0; ia < a.n_a; ++ia) {
        const Real s = dx * cs[2 * ia] + dy * cs[2 * ia + 1];
        Real pc, ps;
        M::cis_rev(kr * s, pc, ps);
        if (lossy) {
          const Real m = M::exp2_(ki * s);
          pc *= m;
          ps *= m;
        }
        const Real* fa = f + ia * 6;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          in[2 * c] += fa[2 * c] * pc - fa[2 * c + 1] * ps;
          in[2 * c + 1] += fa[2 * c] * ps + fa[2 * c + 1] * pc;
        }
      }
      Real zc, zs;
      z_phase(kzd, dz, zc, zs);
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        acc[2 * c] += (double)(in[2 * c] * zc - in[2 * c + 1] * zs);
        acc[2 * c + 1] += (double)(in[2 * c] * zs + in[2 * c + 1] * zc);
      }
    }
  }
  if (active) {
    double2* part = a.part + (size_t)3 * blockIdx.y * a.n_pts + p;
#pragma unroll
    for (int c = 0; c < 3; ++c) part[c * a.n_pts] = make_double2(acc[2 * c], acc[2 * c + 1]);
  }
}

// out[c][idx[j]] = sum of the kappa ranges' fields in order
__global__ void pwe_gather_kernel(const double2* __restrict__ part, int splits, int64_t n, const int* __restrict__ idx,
                                  double2* out) {
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= 3 * n) return;
  double re = 0, im = 0;
#pragma unroll 4
  for (int q = 0; q < splits; ++q) {
    const double2 v = part[(int64_t)q * 3 * n + j];
    re += v.x;
    im += v.y;
  }
  const int64_t c = j / n;
  out[c * n + idx[j - c * n]] = make_double2(re, im);
}

struct PwePoint {
  double x[3];
  int64_t index;
};

// Recursive median split of the points [b, e) into leaves of at most kLeaf
// points, along the wider in-plane extent, along z only where that is 64 times
// the wider: the harmonics kernel's work grows with the in-plane radius of a
// leaf, its height costs nothing.
void split_leaves(PwePoint* pt, int64_t b, int64_t e, std::vector<int>& bounds) {
  if (e - b <= kLeaf) {
    bounds.push_back((int)e);
    return;
  }
  double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
  for (int64_t j = b; j < e; ++j)
    for (int d = 0; d < 3; ++d) {
      lo[d] = std::min(lo[d], pt[j].x[d]);
      hi[d] = std::max(hi[d], pt[j].x[d]);
    }
  int dim = hi[1] - lo[1] > hi[0] - lo[0] ? 1 : 0;
  if (hi[2] - lo[2] > 64.0 * (hi[dim] - lo[dim])) dim = 2;
  // split at a multiple of the leaf size so leaves stay full
  const int64_t half = ((e - b + 1) / 2 + kLeaf - 1) / kLeaf * kLeaf;
  const int64_t mid = std::min(e - 1, b + half);
  std::nth_element(pt + b, pt + mid, pt + e, [&](const PwePoint& u, const PwePoint& v) { return u.x[dim] < v.x[dim]; });
  split_leaves(pt, b, mid, bounds);
  split_leaves(pt, mid, e, bounds);
}

// Points that share (x, y) with at least kColumn others on average (vertical
// cuts) go into leaves of one column each, whose expansion ends at order 0;
// pt is reordered and the leaf bounds appended. false (pt as it was): too few
// of them.
constexpr int kColumn = 16;
bool column_leaves(std::vector<PwePoint>& pt, std::vector<int>& bounds) {
  const int64_t n = (int64_t)pt.size(), most = n / kColumn;
  if (most < 1) return false;
  int64_t size = 16;
  while (size < 4 * most) size *= 2;
  std::vector<int> table(size, -1), column(n);  // hash slots: column numbers
  std::vector<int64_t> first, count;            // a point of the column, its points
  for (int64_t j = 0; j < n; ++j) {
    const double x = pt[j].x[0] + 0.0, y = pt[j].x[1] + 0.0;  // (-0 is 0)
    uint64_t hx, hy;
    std::memcpy(&hx, &x, 8);
    std::memcpy(&hy, &y, 8);
    uint64_t h = (hx ^ (hy * 0x9e3779b97f4a7c15ull)) * 0xd6e8feb86659fd93ull;
    int64_t slot = (int64_t)((h ^ (h >> 32)) & (uint64_t)(size - 1));
    for (;; slot = (slot + 1) & (size - 1)) {
      const int c = table[slot];
      if (c < 0) {
        if ((int64_t)first.size() == most) return false;
        table[slot] = (int)first.size();
        column[j] = (int)first.size();
        first.push_back(j);
        count.push_back(1);
        break;
      }
      if (pt[first[c]].x[0] == pt[j].x[0] && pt[first[c]].x[1] == pt[j].x[1]) {
        column[j] = c;
        ++count[c];
        break;
      }
    }
  }
  std::vector<int64_t> at(first.size());
  int64_t pos = 0;
  for (size_t c = 0; c < first.size(); ++c) {
    at[c] = pos;
    for (int64_t p = 0; p < count[c]; p += kLeaf) bounds.push_back((int)(pos + std::min<int64_t>(p + kLeaf, count[c])));
    pos += count[c];
  }
  std::vector<PwePoint> sorted(n);
  for (int64_t j = 0; j < n; ++j) sorted[at[column[j]]++] = pt[j];
  pt.swap(sorted);
  return true;
}

}  // namespace

extern "C" int smh_pwe_field(smh_ctx* ctx, int kind, int64_t n_k, const double* kp, const double* kz, int64_t n_a,
                             const double* alpha, const double* g, double k_re, double k_im, int64_t n_pts,
                             const double* xyz, double* out, int precision, double* kernel_ms) {
  if (!ctx) return SMH_ERR_ARG;
  SMH_CHECK(ctx, kind == 0 || kind == 1, SMH_ERR_ARG, "kind must be 0 (E) or 1 (omega H)");
  SMH_CHECK(ctx, n_k >= 1 && n_a >= 1 && n_pts >= 0 && kp && kz && alpha && g, SMH_ERR_ARG, "invalid PWE arguments");
  SMH_CHECK(ctx, precision == SMH_FP32 || precision == SMH_FP64, SMH_ERR_ARG, "invalid precision %d", precision);
  SMH_CHECK(ctx, n_pts < (1 << 30) && n_k * n_a < (1 << 30), SMH_ERR_ARG, "PWE too large");
  if (kernel_ms) *kernel_ms = 0.0;
  if (n_pts == 0) return SMH_OK;
  SMH_CHECK(ctx, xyz && out, SMH_ERR_ARG, "points / output are NULL");
  SMH_HIP(ctx, hipSetDevice(ctx->device));
  typedef std::complex<double> zd;
  const zd kk(k_re, k_im);
  SMH_CHECK(ctx, std::abs(kk) > 0, SMH_ERR_ARG, "wavenumber is zero");
  // weights: trapezoid over alpha (inner) and over kappa with the kappa factor (outer);
  // a single kappa sample is a discrete plane wave: its first alpha sample, weight 1
  std::vector<zd> wk(n_k);
  std::vector<double> wa(n_a);
  if (n_k == 1) {
    wk[0] = 1.0;
    std::fill(wa.begin(), wa.end(), 0.0);
    wa[0] = 1.0;
  } else {
    auto KP = [&](int64_t j) { return zd(kp[2 * j], kp[2 * j + 1]); };
    for (int64_t j = 0; j < n_k; ++j) {
      const zd d = (j + 1 < n_k ? KP(j + 1) : KP(j)) - (j > 0 ? KP(j - 1) : KP(j));
      wk[j] = 0.5 * d * KP(j);
    }
    for (int64_t j = 0; j < n_a; ++j)
      wa[j] = n_a == 1 ? 0.0 : 0.5 * ((j + 1 < n_a ? alpha[j + 1] : alpha[j]) - (j > 0 ? alpha[j - 1] : alpha[j]));
  }
  // leaves and their origins; z origin on the side toward which every term decays
  std::vector<PwePoint> pt(n_pts);
  for (int64_t j = 0; j < n_pts; ++j) pt[j] = {{xyz[3 * j], xyz[3 * j + 1], xyz[3 * j + 2]}, j};
  std::vector<int> bounds{0};
  if (!column_leaves(pt, bounds)) split_leaves(pt.data(), 0, n_pts, bounds);
  const int n_leaves = (int)bounds.size() - 1;
  bool up = true, down = true;
  double kmax = 0.0, kim = 0.0;
  for (int64_t k = 0; k < n_k; ++k) {
    if (kz[2 * k + 1] < 0) up = false;
    if (kz[2 * k + 1] > 0) down = false;
    kmax = std::max(kmax, std::hypot(kp[2 * k], kp[2 * k + 1]));
    kim = std::max(kim, std::fabs(kp[2 * k + 1]));
  }
  // device buffers; the first kUp of them are one block, filled here and uploaded in one copy (each copy of a few KB
  // takes a call as long as a kernel)
  enum { KP, KZ, WK, CA, SA, WA, AL, PTS, ORG, LEAF, IDX, LIST, kUp, F_ = kUp, OUT, PART, G_, TRIG, N_BUF };
  size_t sizes[N_BUF], up_off[kUp + 1] = {0};
  sizes[KP] = sizes[KZ] = sizes[WK] = (size_t)n_k * 16;
  sizes[CA] = sizes[SA] = sizes[WA] = sizes[AL] = (size_t)n_a * 8;
  sizes[PTS] = (size_t)3 * n_pts * 8;
  sizes[ORG] = (size_t)4 * n_leaves * 8;
  sizes[LEAF] = bounds.size() * 4;
  sizes[IDX] = (size_t)n_pts * 4;
  sizes[LIST] = (size_t)n_leaves * 4;
  for (int i = 0; i < kUp; ++i) up_off[i + 1] = up_off[i] + (sizes[i] + 15) / 16 * 16;
  std::vector<double> block(up_off[kUp] / 8);
  auto in = [&](int i) { return block.data() + up_off[i] / 8; };
  std::memcpy(in(KP), kp, sizes[KP]);
  std::memcpy(in(KZ), kz, sizes[KZ]);
  std::memcpy(in(WK), wk.data(), sizes[WK]);
  std::memcpy(in(WA), wa.data(), sizes[WA]);
  std::memcpy(in(AL), alpha, sizes[AL]);
  std::memcpy(in(LEAF), bounds.data(), sizes[LEAF]);
  for (int64_t j = 0; j < n_a; ++j) {
    in(CA)[j] = std::cos(alpha[j]);
    in(SA)[j] = std::sin(alpha[j]);
  }
  double *pts = in(PTS), *org = in(ORG);
  int* idx = (int*)in(IDX);
  // leaves by kernel: order 0, harmonics with up to 31 orders, up to 63, one term per azimuth. The harmonics pay where
  // their orders (about 20 instructions each, and most kappa have fewer than the largest) are below half the
  // azimuths (26 instructions and three or four transcendental ones each); growth of e^{|Im kappa| rho} would
  // cost digits in the orders' sum, so lossy contours keep |Im kappa| R below 1.
  constexpr int kKernels = 4;
  std::vector<int> list[kKernels];
  for (int l = 0; l < n_leaves; ++l) {
    double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
    for (int j = bounds[l]; j < bounds[l + 1]; ++j) {
      idx[j] = (int)pt[j].index;
      for (int d = 0; d < 3; ++d) {
        pts[3 * (size_t)j + d] = pt[j].x[d];
        lo[d] = std::min(lo[d], pt[j].x[d]);
        hi[d] = std::max(hi[d], pt[j].x[d]);
      }
    }
    double* o = &org[4 * (size_t)l];
    o[0] = 0.5 * (lo[0] + hi[0]);
    o[1] = 0.5 * (lo[1] + hi[1]);
    o[2] = up ? lo[2] : (down ? hi[2] : 0.5 * (lo[2] + hi[2]));
    double r2 = 0.0;
    for (int j = bounds[l]; j < bounds[l + 1]; ++j) {
      const double dx = pt[j].x[0] - o[0], dy = pt[j].x[1] - o[1];
      r2 = std::max(r2, dx * dx + dy * dy);
    }
    o[3] = std::sqrt(r2);
    const int m = max_order(precision, kmax * o[3]);
    const bool harmonics = m >= 0 && 2 * m <= n_a && kim * o[3] <= 1.0;
    list[!harmonics ? 3 : (m == 0 ? 0 : (precision == SMH_FP32 && m < 32 ? 1 : 2))].push_back(l);
  }
  // kappa ranges: about eight workgroups per CU, no more ranges than 16s of kappa, whole eights of kappa each (the
  // last one what is left)
  const int want = (int)std::max<int64_t>(1, std::min<int64_t>((8 * (int64_t)ctx->num_cu + n_leaves - 1) / n_leaves,
                                                               (n_k + 15) / 16));
  const int per_split = (int)((n_k + want - 1) / want + 7) / 8 * 8;
  const int splits = (int)((n_k + per_split - 1) / per_split);
  // device buffers
  const size_t rs = precision == SMH_FP32 ? sizeof(float) : sizeof(double);
  const int kc = (int)std::max<int64_t>(1, std::min<int64_t>(16, (48 * 1024) / (n_a * 6 * (int64_t)rs)));
  const size_t lds = (size_t)2 * n_a * rs + (size_t)kc * n_a * 6 * rs;
  SMH_CHECK(ctx, lds <= 160 * 1024, SMH_ERR_UNSUPPORTED, "too many azimuth samples (%lld)", (long long)n_a);
  const int trig_rows = (int)(n_a + 3) / 4 * 4;
  const bool harmonic = !list[1].empty() || !list[2].empty();
  int* order = (int*)in(LIST);
  for (const std::vector<int>& l : list) order = std::copy(l.begin(), l.end(), order);
  const size_t waves = (size_t)n_k * n_a;
  sizes[F_] = 3 * waves * 16;
  sizes[OUT] = (size_t)3 * n_pts * 16;
  sizes[PART] = splits * sizes[OUT];
  sizes[G_] = 2 * waves * 16;
  sizes[TRIG] = harmonic ? (size_t)trig_rows * 2 * (kMaxM + 1) * rs : 0;
  char* d_up = nullptr;
  void* buf[N_BUF] = {nullptr};
  auto release = [&]() {
    if (d_up) (void)hipFree(d_up);
    for (int i = kUp; i < N_BUF; ++i)
      if (buf[i]) (void)hipFree(buf[i]);
  };
  bool ok = hipMalloc(&d_up, up_off[kUp]) == hipSuccess;
  for (int i = 0; i < kUp && ok; ++i) buf[i] = d_up + up_off[i];
  for (int i = kUp; i < N_BUF && ok; ++i) ok = sizes[i] == 0 || hipMalloc(&buf[i], sizes[i]) == hipSuccess;
  if (!ok) {
    release();
    return smh_fail(ctx, SMH_ERR_HIP, "PWE device allocation failed");
  }
  hipStream_t s = ctx->stream;
  if (hipMemcpyAsync(d_up, block.data(), up_off[kUp], hipMemcpyHostToDevice, s) != hipSuccess ||
      hipMemcpyAsync(buf[G_], g, sizes[G_], hipMemcpyHostToDevice, s) != hipSuccess) {
    release();
    return smh_fail(ctx, SMH_ERR_HIP, "PWE upload failed");
  }
  PweArgs a;
  a.F = (const double2*)buf[F_];
  a.kp = (const double2*)buf[KP];
  a.kz = (const double2*)buf[KZ];
  a.ca = (const double*)buf[CA];
  a.sa = (const double*)buf[SA];
  a.trig = buf[TRIG];
  a.pts = (const double*)buf[PTS];
  a.leaf = (const int*)buf[LEAF];
  a.org = (const double*)buf[ORG];
  a.part = (double2*)buf[PART];
  a.n_pts = n_pts;
  a.n_k = (int)n_k;
  a.n_a = (int)n_a;
  a.kc = kc;
  a.per_split = per_split;
  void* fn[kKernels] = {precision == SMH_FP32 ? reinterpret_cast<void*>(&pwe_column_kernel<float>)
                                              : reinterpret_cast<void*>(&pwe_column_kernel<double>),
                        reinterpret_cast<void*>(&pwe_harmonics_kernel<float, 8>),
                        precision == SMH_FP32 ? reinterpret_cast<void*>(&pwe_harmonics_kernel<float, 4>)
                                              : reinterpret_cast<void*>(&pwe_harmonics_kernel<double, 4>),
                        precision == SMH_FP32 ? reinterpret_cast<void*>(&pwe_field_kernel<float>)
                                              : reinterpret_cast<void*>(&pwe_field_kernel<double>)};
  hipError_t e = hipFuncSetAttribute(fn[3], hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e == hipSuccess) e = hipEventRecord(ctx->ev0, s);
  if (e == hipSuccess) {
    hipLaunchKernelGGL(pwe_coefficients_kernel, dim3((unsigned)((waves + 255) / 256)), dim3(256), 0, s, kind, (int)n_k,
                       (int)n_a, (const double2*)buf[G_], a.kp, a.kz, a.ca, a.sa, (const double2*)buf[WK],
                       (const double*)buf[WA], make_double2(k_re, k_im), (double2*)buf[F_]);
    const unsigned tb = (unsigned)((trig_rows * (kMaxM + 1) + 255) / 256);
    if (!harmonic)
      ;  // (only the harmonics read it)
    else if (precision == SMH_FP32)
      hipLaunchKernelGGL(pwe_trig_kernel<float>, dim3(tb), dim3(256), 0, s, (int)n_a, trig_rows, (const double*)buf[AL],
                         (float*)buf[TRIG]);
    else
      hipLaunchKernelGGL(pwe_trig_kernel<double>, dim3(tb), dim3(256), 0, s, (int)n_a, trig_rows,
                         (const double*)buf[AL], (double*)buf[TRIG]);
    e = hipGetLastError();
  }
  size_t at = 0;
  for (int i = 0; i < kKernels && e == hipSuccess; ++i) {
    if (list[i].empty()) continue;
    a.list = (const int*)buf[LIST] + at;
    at += list[i].size();
    void* args[] = {&a};
    e = hipLaunchKernel(fn[i], dim3((unsigned)list[i].size(), (unsigned)splits), dim3(256), args, i == 3 ? lds : 0, s);
  }
  if (e == hipSuccess) {
    hipLaunchKernelGGL(pwe_gather_kernel, dim3((unsigned)((3 * n_pts + 255) / 256)), dim3(256), 0, s,
                       (const double2*)buf[PART], splits, n_pts, (const int*)buf[IDX], (double2*)buf[OUT]);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipEventRecord(ctx->ev1, s);
  if (e == hipSuccess) e = hipMemcpyAsync(out, buf[OUT], sizes[OUT], hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  float ms = 0;
  if (e == hipSuccess) e = hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1);
  release();
  SMH_CHECK(ctx, e == hipSuccess, SMH_ERR_HIP, "PWE field kernel failed: %s", hipGetErrorString(e));
  if (kernel_ms) *kernel_ms = ms;
  return SMH_OK;
}

// ---- plane wave expansion of the scattered field --------------------------
// g_dir(pol, kappa, alpha) = sum_p e^{-i kappa (x_p cos a + y_p sin a)} e^{i kz_dir (z_ref - z_p)}
//                            * sum_m e^{i m a} c_{p,m,pol,dir}(kappa),
// c_{p,m,pol,dir} = sum_{tau,l} b_{p,tau l m} B_{tau l m,pol}(+-kz/k, kappa/k) / (2 pi kz k)
// (swe_to_pwe_conversion, fields/transformations.py:133-226, summed over the
// particles of one layer as scattered_field_pwe, postprocessing/scattered_field.py:80-150).
// Per kappa this is a complex matrix product over the particles, phases
// [alpha][particle] times coefficients [particle][(m, pol, dir)], on the MFMA
// 16x16x4 (FP32 or FP64): a wave holds kAsmTiles tiles of 16 alpha, its lanes
// compute one phase each per four particles (no phase twice), and the
// coefficients of a chunk of particles, e^{+-i kz (z_ref - z)} included, are
// staged in LDS by the workgroup. The phase's argument is formed and reduced to
// a revolution in FP64 (FP32: then native sine and cosine). The particles are
// split over workgroups until the chip is filled (a far field of 90 polar
// angles, or the one direction of an extinction cross section, has too few
// kappa for that); a second kernel adds the splits' sums in FP64. Bound by the
// FP64 sincos of the phases (about 60 instructions per particle and alpha)
// beside as much time in the MFMA: 90 x 361 waves, 1000 particles, l_max 3, FP64:
// 1.34 ms when a thread summed all orders of one alpha in registers.
// The MFMA's sums go through the sum over m into FP64 ones every kAsmFlush particles:
// where the waves alone fill the chip, one workgroup sums all particles, and one
// running FP32 sum of 10000 of them is off by 2.5e-6 (1000 x 361 waves over 60 um,
// 15.3 ms), in this form by 3.0e-7 (16.7 ms). FP64, 2000 particles: 6.6 -> 6.8 ms.
// A launch covers kAsmOrders orders m at most; more run as several launches,
// each adding its orders' share into g.
namespace {

constexpr int kAsmChunk = 32;   // particles staged at a time
constexpr int kAsmFlush = 4 * kAsmChunk;  // particles of one sum on the MFMA
constexpr int kAsmTiles = 2;    // alpha tiles per wave
constexpr int kAsmWaves = 4;
constexpr int kAsmOrders = 12;  // orders per launch: 4 (dir, pol) each in 3 column tiles

struct AsmArgs {
  const double* pts;    // [n_part][3]
  const double2* coef;  // [n_part][B]
  const double2* kp;    // [n_k]
  const double2* kz;    // [n_k] upgoing kz
  const double2* btab;  // [n_k][2 dir][2 pol][B], 1 / (2 pi kz k) included
  const int* nlist;     // [NM][LM] multipole indices n of order m = j + m_first (-1: none)
  const double* alpha;  // [n_a]
  double2* part;        // [splits][2 dir][2 pol][n_k][n_a]
  double z_ref;
  int64_t n_part;
  int B, LM, NM, n_k, n_a;
  int per_split;        // particles per blockIdx.y
  unsigned a_blocks;    // alpha blocks per kappa (blockIdx.x = kappa * a_blocks + block)
  int m_first;          // order of the launch's first row of nlist
};

// CT: tiles of 16 columns (m, q), q = (dir, pol), of the real and of the imaginary parts
template <typename Real, int CT>
__global__ void __launch_bounds__(64 * kAsmWaves, sizeof(Real) == 4 ? 3 : 2) pwe_assemble_kernel(AsmArgs a) {
  using M = smh::Mfma<Real>;
  constexpr int Q = 4, SC = CT * 16 + 16;  // (the row stride puts neighbouring particles in other banks)
  __shared__ Real cr[kAsmChunk][SC], ci[kAsmChunk][SC];
  __shared__ double px[kAsmChunk], py[kAsmChunk];
  __shared__ double2 ez[kAsmChunk][2];
  __shared__ double2 em[kAsmWaves][kAsmTiles * 16][4 * CT];  // e^{i m alpha}, each wave's alphas and all orders
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, c = lane & 15, h = lane >> 4;
  const int k = (int)(blockIdx.x / a.a_blocks), ab = (int)(blockIdx.x - k * a.a_blocks);
  const int tile0 = (ab * (int)(blockDim.x >> 6) + wave) * kAsmTiles;
  const double2 kp = a.kp[k], kz = a.kz[k];
  const Turns kturn = turns_of(-kp.x);        // e^{-i kappa s}
  const double klog = kp.y * kLog2e;          // |e^{-i kappa s}| = 2^(klog s)
  const bool lossy = kp.y != 0.0;
  // this lane's alpha of each tile
  double ca[kAsmTiles], sa[kAsmTiles];
#pragma unroll
  for (int t = 0; t < kAsmTiles; ++t) {
    const int ia = (tile0 + t) * 16 + c;
    sincos(ia < a.n_a ? a.alpha[ia] : 0.0, &sa[t], &ca[t]);
  }
  typename M::v4 ar[kAsmTiles][CT], ai[kAsmTiles][CT];
#pragma unroll
  for (int t = 0; t < kAsmTiles; ++t)
#pragma unroll
    for (int j = 0; j < CT; ++j) ar[t][j] = ai[t][j] = typename M::v4{0, 0, 0, 0};
  for (int w = lane; w < kAsmTiles * 16 * 4 * CT; w += 64) {
    const int r = w / (4 * CT), m = w - r * (4 * CT), ia = tile0 * 16 + r;
    double es, ec;
    sincos((double)(m + a.m_first) * (ia < a.n_a ? a.alpha[ia] : 0.0), &es, &ec);
    em[wave][r][m] = make_double2(ec, es);
  }
  // the lane's share (its columns' orders) of the sum over m of e^{i m alpha}, and the running sums cleared
  double gr[kAsmTiles][4], gi[kAsmTiles][4];
#pragma unroll
  for (int t = 0; t < kAsmTiles; ++t)
#pragma unroll
    for (int v = 0; v < 4; ++v) gr[t][v] = gi[t][v] = 0.0;
  auto flush = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < kAsmTiles; ++t)
#pragma unroll
      for (int j = 0; j < CT; ++j) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const double2 e = em[wave][t * 16 + (M::kRowIs4q ? 4 * h + v : 4 * v + h)][4 * j + (c >> 2)];
          const double re = (double)ar[t][j][v], im = (double)ai[t][j][v];
          gr[t][v] += re * e.x - im * e.y;
          gi[t][v] += re * e.y + im * e.x;
        }
        ar[t][j] = ai[t][j] = typename M::v4{0, 0, 0, 0};
      }
  };
  const int64_t first = (int64_t)blockIdx.y * a.per_split;
  const int64_t last = first + a.per_split < a.n_part ? first + a.per_split : a.n_part;
  for (int64_t p0 = first; p0 < last; p0 += kAsmChunk) {
    const int np = (int)(last - p0 < kAsmChunk ? last - p0 : kAsmChunk);
    __syncthreads();
    for (int p = tid; p < kAsmChunk; p += blockDim.x) {
      const bool on = p < np;
      px[p] = on ? a.pts[3 * (p0 + p)] : 0.0;
      py[p] = on ? a.pts[3 * (p0 + p) + 1] : 0.0;
      // e^{i kz (z_ref - z_p)} (up) and e^{-i kz (z_ref - z_p)} (down)
      const double dz = on ? a.z_ref - a.pts[3 * (p0 + p) + 2] : 0.0;
      double su, cu;
      sincos(kz.x * dz, &su, &cu);
      const double mu = exp(-kz.y * dz), md = exp(kz.y * dz);
      ez[p][0] = make_double2(mu * cu, mu * su);
      ez[p][1] = make_double2(md * cu, -md * su);
    }
    __syncthreads();
    for (int w = tid; w < kAsmChunk * CT * 16; w += blockDim.x) {
      const int p = w / (CT * 16), col = w - p * (CT * 16), m = col >> 2, q = col & 3;
      double re = 0, im = 0;
      if (p < np && m < a.NM) {
        for (int j = 0; j < a.LM; ++j) {
          const int n = a.nlist[m * a.LM + j];
          if (n < 0) break;
          const double2 b = a.coef[(p0 + p) * a.B + n], t = a.btab[((size_t)k * Q + q) * a.B + n];
          re += b.x * t.x - b.y * t.y;
          im += b.x * t.y + b.y * t.x;
        }
        const double2 e = ez[p][q >> 1];
        const double r = re * e.x - im * e.y;
        im = re * e.y + im * e.x;
        re = r;
      }
      cr[p][col] = (Real)re;
      ci[p][col] = (Real)im;
    }
    __syncthreads();
    if (tile0 * 16 >= a.n_a) continue;
    if (p0 > first && (p0 - first) % kAsmFlush == 0) flush();
    for (int s = 0; s < (np + 3) / 4; ++s) {
      const int p = 4 * s + h;  // (particles beyond np have zero coefficients)
      Real br[CT], bi[CT];
#pragma unroll
      for (int j = 0; j < CT; ++j) {
        br[j] = cr[p][16 * j + c];
        bi[j] = ci[p][16 * j + c];
      }
#pragma unroll
      for (int t = 0; t < kAsmTiles; ++t) {
        const double sd = px[p] * ca[t] + py[p] * sa[t];
        Real pr, pi;
        cis_turns(turn_fraction(kturn, sd), pr, pi);
        if (lossy) {
          const Real mg = exp2_split(klog * sd, Real(0));
          pr *= mg;
          pi *= mg;
        }
#pragma unroll
        for (int j = 0; j < CT; ++j) {
          ar[t][j] = M::op(pr, br[j], ar[t][j]);
          ai[t][j] = M::op(pr, bi[j], ai[t][j]);
          ar[t][j] = M::op(pi, -bi[j], ar[t][j]);
          ai[t][j] = M::op(pi, br[j], ai[t][j]);
        }
      }
    }
  }
  flush();
  // the lanes of the same q
#pragma unroll
  for (int t = 0; t < kAsmTiles; ++t)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int ia = (tile0 + t) * 16 + (M::kRowIs4q ? 4 * h + v : 4 * v + h);
#pragma unroll
      for (int off = 4; off < 16; off <<= 1) {
        gr[t][v] += __shfl_xor(gr[t][v], off);
        gi[t][v] += __shfl_xor(gi[t][v], off);
      }
      if (c < Q && ia < a.n_a)
        a.part[(((size_t)blockIdx.y * Q + c) * a.n_k + k) * a.n_a + ia] = make_double2(gr[t][v], gi[t][v]);
    }
}

// g = sum of the splits in order (g += it for the later launches of a chunked order range)
__global__ void pwe_sum_kernel(const double2* __restrict__ part, int splits, int64_t count, int accumulate,
                               double2* g) {
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= count) return;
  double2 s = accumulate ? g[j] : make_double2(0.0, 0.0);
#pragma unroll 4
  for (int q = 0; q < splits; ++q) {
    const double2 v = part[q * count + j];
    s.x += v.x;
    s.y += v.y;
  }
  g[j] = s;
}

template <typename Real>
void* assemble_kernel_for(int nm) {
  switch ((4 * nm + 15) / 16) {
    case 1: return reinterpret_cast<void*>(&pwe_assemble_kernel<Real, 1>);
    case 2: return reinterpret_cast<void*>(&pwe_assemble_kernel<Real, 2>);
    default: return reinterpret_cast<void*>(&pwe_assemble_kernel<Real, 3>);
  }
}

}  // namespace

extern "C" int smh_pwe_assemble(smh_ctx* ctx, int64_t n_part, const double* xyz, int l_max, int m_max,
                                const double* coef, double z_ref, int64_t n_k, const double* kp, const double* kz,
                                const double* btab, int64_t n_a, const double* alpha, double* g, int precision,
                                double* kernel_ms) {
  if (!ctx) return SMH_ERR_ARG;
  SMH_CHECK(ctx, n_part >= 1 && xyz && coef && kp && kz && btab && alpha && g, SMH_ERR_ARG,
            "invalid PWE assembly arguments");
  SMH_CHECK(ctx, l_max >= 1 && m_max >= 1 && m_max <= l_max && l_max <= 64, SMH_ERR_ARG,
            "invalid l_max %d / m_max %d", l_max, m_max);
  SMH_CHECK(ctx, n_k >= 1 && n_a >= 1 && n_k < (1 << 30) && n_a < (1 << 30) && n_part < (1 << 30), SMH_ERR_ARG,
            "invalid sizes");
  SMH_CHECK(ctx, precision == SMH_FP32 || precision == SMH_FP64, SMH_ERR_ARG, "invalid precision %d", precision);
  if (kernel_ms) *kernel_ms = 0.0;
  SMH_HIP(ctx, hipSetDevice(ctx->device));
  const int B = smh_blocksize(l_max, m_max), n_orders = 2 * m_max + 1, LM = 2 * l_max;
  // orders per launch: all of them when they fit, else chunks of kAsmOrders
  // (the last one padded with empty orders, whose rows of nlist hold -1)
  const int NM = n_orders <= kAsmOrders ? n_orders : kAsmOrders;
  const int n_chunks = (n_orders + NM - 1) / NM;
  // multipole indices of each order m (row j: order j - m_max)
  std::vector<int> nlist((size_t)n_chunks * NM * LM, -1), fill(n_chunks * NM, 0);
  for (int tau = 0; tau < 2; ++tau)
    for (int l = 1; l <= l_max; ++l) {
      const int ml = std::min(l, m_max);
      for (int m = -ml; m <= ml; ++m) {
        const int j = m + m_max;
        nlist[(size_t)j * LM + fill[j]++] = smh_multi_to_single(tau, l, m, l_max, m_max);
      }
    }
  // waves of a workgroup: no more than the alpha tiles ask for
  const int64_t tiles = (n_a + 15) / 16;
  const int waves = (int)std::min<int64_t>(kAsmWaves, (tiles + kAsmTiles - 1) / kAsmTiles);
  const int threads = 64 * waves;
  const unsigned a_blocks = (unsigned)((tiles + waves * kAsmTiles - 1) / (waves * kAsmTiles));
  // splits of the particles: about eight workgroups per CU, whole chunks each
  const int64_t blocks = n_k * a_blocks, chunks = (n_part + kAsmChunk - 1) / kAsmChunk;
  const int64_t want = std::max<int64_t>(1, std::min<int64_t>((8 * (int64_t)ctx->num_cu + blocks - 1) / blocks, chunks));
  const int per_split = (int)((chunks + want - 1) / want) * kAsmChunk;
  const int splits = (int)((n_part + per_split - 1) / per_split);
  const int64_t count = 4 * n_k * n_a;
  SMH_CHECK(ctx, blocks < ((int64_t)1 << 31), SMH_ERR_ARG, "invalid sizes");
  void* buf[9] = {nullptr};
  const size_t sizes[9] = {(size_t)n_part * 24, (size_t)n_part * B * 16, (size_t)n_k * 16, (size_t)n_k * 16,
                           (size_t)n_k * 4 * B * 16, nlist.size() * 4, (size_t)n_a * 8, (size_t)count * 16,
                           (size_t)splits * count * 16};
  auto release = [&]() {
    for (void* b : buf)
      if (b) hipFree(b);
  };
  for (int i = 0; i < 9; ++i)
    if (hipMalloc(&buf[i], sizes[i]) != hipSuccess) {
      release();
      return smh_fail(ctx, SMH_ERR_HIP, "PWE assembly allocation failed");
    }
  hipStream_t s = ctx->stream;
  const void* src[7] = {xyz, coef, kp, kz, btab, nlist.data(), alpha};
  for (int i = 0; i < 7; ++i)
    if (hipMemcpyAsync(buf[i], src[i], sizes[i], hipMemcpyHostToDevice, s) != hipSuccess) {
      release();
      return smh_fail(ctx, SMH_ERR_HIP, "PWE assembly upload failed");
    }
  AsmArgs a;
  a.pts = (const double*)buf[0];
  a.coef = (const double2*)buf[1];
  a.kp = (const double2*)buf[2];
  a.kz = (const double2*)buf[3];
  a.btab = (const double2*)buf[4];
  a.alpha = (const double*)buf[6];
  a.part = (double2*)buf[8];
  a.per_split = per_split;
  a.a_blocks = a_blocks;
  a.z_ref = z_ref;
  a.n_part = n_part;
  a.B = B;
  a.LM = LM;
  a.NM = NM;
  a.n_k = (int)n_k;
  a.n_a = (int)n_a;
  void* kfn = precision == SMH_FP32 ? assemble_kernel_for<float>(NM) : assemble_kernel_for<double>(NM);
  hipError_t e = hipEventRecord(ctx->ev0, s);
  void* args[] = {&a};
  for (int c = 0; c < n_chunks && e == hipSuccess; ++c) {
    a.nlist = (const int*)buf[5] + (size_t)c * NM * LM;
    a.m_first = c * NM - m_max;
    e = hipLaunchKernel(kfn, dim3((unsigned)blocks, (unsigned)splits), dim3(threads), args, 0, s);
    if (e != hipSuccess) break;
    hipLaunchKernelGGL(pwe_sum_kernel, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, s,
                       (const double2*)buf[8], splits, count, c > 0 ? 1 : 0, (double2*)buf[7]);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipEventRecord(ctx->ev1, s);
  if (e == hipSuccess) e = hipMemcpyAsync(g, buf[7], sizes[7], hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  float ms = 0;
  if (e == hipSuccess) e = hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1);
  release();
  SMH_CHECK(ctx, e == hipSuccess, SMH_ERR_HIP, "PWE assembly kernel failed: %s", hipGetErrorString(e));
  if (kernel_ms) *kernel_ms = ms;
  return SMH_OK;
}
