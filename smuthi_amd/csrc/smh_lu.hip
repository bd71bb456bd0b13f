// Direct solve of (1 - T W) b = T a for the explicit operator: the
// solver_type='LU' branch of LinearSystem.solve (linearsystem/linear_system.py:
// 259-268), which factors the stored master matrix once with LAPACK
// (scipy lu_factor), keeps the factors and solves every right-hand side with
// them (lu_solve). Here the master matrix M = 1 - diag(t) W is formed in FP64
// from the device-resident explicit matrix, factored with partial pivoting (up
// to 2048 unknowns by lu_step_kernel, beyond by rocSOLVER's getrf) and solved by
// getrs, all on the device; the factors stay
// on the operator for later right-hand sides with the same T. Every solution
// is certified by its FP64 residual ||b - M x|| / ||b||, computed with the
// explicit matvec.
//
// The explicit matrix is row-major on the padded index (i * B + n), which
// rocSOLVER (column-major) sees as M^T: getrf factors that matrix and getrs
// solves with its transpose, i.e. with M itself. Padding slots carry t = 0, so
// their rows and columns of M are those of the identity.
#include <rocblas/rocblas.h>
#include <rocsolver/rocsolver.h>

#include <chrono>
#include <cmath>

#include "smh_op.h"

namespace {

int blocks_of(int64_t n, int t = 256) { return (int)std::min<int64_t>((n + t - 1) / t, 1 << 20); }

// M = I - diag(t) W on the padded index, row-major [n][n], or (unit 0) M - I
__global__ void master_dense_kernel(const double2* __restrict__ W, const double2* __restrict__ t, int64_t n, double unit,
                                    double2* __restrict__ M) {
  const int64_t total = n * n;
  for (int64_t f = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; f < total; f += (int64_t)gridDim.x * blockDim.x) {
    const int64_t r = f / n, c = f - r * n;
    const double2 w = W[f], a = t[r];
    double re = -(a.x * w.x - a.y * w.y);
    const double im = -(a.x * w.y + a.y * w.x);
    if (r == c) re += unit;
    M[f] = make_double2(re, im);
  }
}

// r = b - (x - t o y) for nrhs padded vectors [nrhs][n] (y = W x); per block
// partial sums of |r|^2 and |b|^2 for each right-hand side
__global__ void residual_parts_kernel(const double2* __restrict__ b, const double2* __restrict__ x,
                                      const double2* __restrict__ y, const double2* __restrict__ t, int64_t n,
                                      double* __restrict__ parts) {
  const int rhs = blockIdx.y;
  __shared__ double red[2][256];
  double rr = 0, bb = 0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t e = (int64_t)rhs * n + i;
    const double2 a = t[i], yv = y[e], xv = x[e], bv = b[e];
    const double mr = xv.x - (a.x * yv.x - a.y * yv.y), mi = xv.y - (a.x * yv.y + a.y * yv.x);
    const double dr = bv.x - mr, di = bv.y - mi;
    rr += dr * dr + di * di;
    bb += bv.x * bv.x + bv.y * bv.y;
  }
  red[0][threadIdx.x] = rr;
  red[1][threadIdx.x] = bb;
  __syncthreads();
  for (int w = blockDim.x / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) {
      red[0][threadIdx.x] += red[0][threadIdx.x + w];
      red[1][threadIdx.x] += red[1][threadIdx.x + w];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    parts[((size_t)rhs * gridDim.x + blockIdx.x) * 2] = red[0][0];
    parts[((size_t)rhs * gridDim.x + blockIdx.x) * 2 + 1] = red[1][0];
  }
}

// ---- factorisation of matrices up to kLuRows * 2 rows ----------------------
// Column-major A(i, j) = A[j n + i], in place, partial pivoting by |re| + |im|
// (first of equals), LAPACK's factors and 1-based pivots. One launch per panel
// of kLuPanel columns: workgroup 0 brings the next panel up to date and
// factors it while the others bring the remaining columns up to date, a strip
// of kLuPanel columns each, and exchange the rows of the columns before.
// Bound by the chain of pivots: a panel's rows stay in the registers of one
// workgroup (two per thread), so that a pivot costs two barriers and no memory
// access. 1800 unknowns (60 spheres, l_max 3): 13.2 ms in some 4000 launches of
// rocSOLVER's getrf, 6.0 ms in 226 launches here, 34 us with two rows per thread
// and 21 with one; solutions' errors against refined ones 4 to 8 % below getrf's
// (spheres, 240 to 1800 unknowns: 4.7e-16 to 7.1e-16). With
// more than 2048 rows the panel no longer fits the registers, and a pass over the matrix per eight columns no
// longer the last-level cache: getrf.
constexpr int kLuPanel = 8, kLuRows = 1024, kLuWaves = kLuRows / 64;

// Row exchanges of a panel, as one permutation of the rows it touches:
// row[t] takes the value of row[src[t]]; row[j] = first column + j, j < width.
// origin[t]: of the row that comes to row[t] (lu_step_kernel).
struct LuPerm {
  int count;
  int row[2 * kLuPanel], src[2 * kLuPanel], origin[2 * kLuPanel];
};

__device__ inline double2 cfma(double2 a, double2 l, double2 u) {  // a + l u
  a.x = fma(l.x, u.x, a.x);
  a.x = fma(-l.y, u.y, a.x);
  a.y = fma(l.x, u.y, a.y);
  a.y = fma(l.y, u.x, a.y);
  return a;
}

// Largest value (of non-negative doubles, by their bits) and smallest index of the row of 16 lanes, in all of them
template <int kCtrl>
__device__ __forceinline__ unsigned dpp(unsigned v) {
  return (unsigned)__builtin_amdgcn_mov_dpp((int)v, kCtrl, 0xF, 0xF, false);
}
template <int kCtrl>
__device__ __forceinline__ unsigned long long max_dpp(unsigned long long k) {
  const unsigned long long o =
      ((unsigned long long)dpp<kCtrl>((unsigned)(k >> 32)) << 32) | dpp<kCtrl>((unsigned)(k & 0xffffffffu));
  return o > k ? o : k;
}
__device__ __forceinline__ unsigned long long max_row(unsigned long long k) {
  k = max_dpp<0x128>(k);  // row_ror:8, 4, 2, 1
  k = max_dpp<0x124>(k);
  k = max_dpp<0x122>(k);
  return max_dpp<0x121>(k);
}
__device__ __forceinline__ unsigned min_row(unsigned i) {
  i = min(i, dpp<0x128>(i));
  i = min(i, dpp<0x124>(i));
  i = min(i, dpp<0x122>(i));
  return min(i, dpp<0x121>(i));
}
__device__ __forceinline__ unsigned long long max_xor(unsigned long long k, int d) {
  const unsigned long long o = __shfl_xor(k, d);
  return o > k ? o : k;
}

__device__ inline double2 csub(double2 a, double2 l, double2 u) {  // a - l u
  a.x = fma(-l.x, u.x, a.x);
  a.x = fma(l.y, u.y, a.x);
  a.y = fma(-l.x, u.y, a.y);
  a.y = fma(-l.y, u.x, a.y);
  return a;
}

// k: first column of the factored panel (strip k / kLuPanel), or -kLuPanel for
// the first launch, which only factors strip 0. Rows below the panel number at
// most R * kLuRows. Block b < gridDim.x takes strip k / kLuPanel + 1 (b = 0,
// if there is one) or one of the others.
// The trailing matrix is kept without the identity of A = I - ..: a row's 1, in
// the column it had before all exchanges (its origin), is added when its
// column's panel is factored or its row becomes one of U. The roundings of
// the updates, one per panel, are then of the coupling's size instead of 1.
// origin: every row's before (in) and after (out) the factored panel's exchanges.
template <int R>
__global__ void __launch_bounds__(kLuRows) lu_step_kernel(double2* __restrict__ A, int64_t n, int k, LuPerm* perms,
                                                          const int* __restrict__ origin_in, int* origin_out,
                                                          int* ipiv, int* info) {
  __shared__ double2 sv[kLuPanel][2 * kLuPanel], us[kLuPanel][kLuPanel], l11[kLuPanel][kLuPanel];
  __shared__ double2 prow[kLuPanel], orow[kLuPanel];
  __shared__ unsigned long long redk[kLuWaves];
  __shared__ unsigned redi[kLuWaves];
  __shared__ int pivots[kLuPanel], origin[2 * kLuRows], moved[2 * kLuPanel];
  const int tid = threadIdx.x, N = (int)n, strips = (N + kLuPanel - 1) / kLuPanel;
  const int sk = k >= 0 ? k / kLuPanel : -1;  // strip of the factored panel
  int strip = sk + 1 < strips ? ((int)blockIdx.x == 0 ? sk + 1 : (int)blockIdx.x - 1) : (int)blockIdx.x;
  if (sk + 1 < strips && blockIdx.x > 0 && strip >= sk) strip += sk >= 0 ? 2 : 1;
  const int c0 = strip * kLuPanel, w = min(kLuPanel, N - c0);
  const int wk = kLuPanel, row0 = k + wk;  // (a panel with strips after it is full)
  double2* C = A + (int64_t)c0 * n;
  if (k >= 0) {
    // row exchanges of the strip
    const LuPerm& pm = perms[sk];
    const int r = tid & (2 * kLuPanel - 1), c = tid / (2 * kLuPanel), count = pm.count;
    const bool mine = c < w && r < count;
    if (mine) sv[c][r] = C[c * n + pm.row[r]];
    if (tid < count) moved[tid] = pm.origin[tid];
    if (strip == sk + 1)
      for (int i = row0 - wk + tid; i < N; i += kLuRows) origin[i] = origin_in[i];
    if (strip > sk && tid < kLuPanel * kLuPanel) {
      const int i = tid / kLuPanel, j = tid % kLuPanel;  // L(j, i) of the panel's triangle
      l11[j][i] = A[(int64_t)(k + i) * n + k + j];
    }
    __syncthreads();
    if (mine && (strip < sk || r >= wk)) C[c * n + pm.row[r]] = sv[c][pm.src[r]];
    if (strip < sk) return;
    // the strip's rows of U
    if (tid < w) {
      double2 u[kLuPanel];
#pragma unroll
      for (int j = 0; j < kLuPanel; ++j) {
        u[j] = sv[tid][pm.src[j]];
        if (moved[j] == c0 + tid) u[j].x += 1.0;
#pragma unroll
        for (int i = 0; i < j; ++i) u[j] = csub(u[j], l11[j][i], u[i]);
        us[j][tid] = u[j];
        C[tid * n + k + j] = u[j];
      }
    }
    __syncthreads();
    if (strip == sk + 1 && tid < count) origin[pm.row[tid]] = moved[tid];
    // the rows below: C -= L U
    double2 l[R][kLuPanel];
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int i = row0 + tid + q * kLuRows;
#pragma unroll
      for (int j = 0; j < kLuPanel; ++j) l[q][j] = i < N ? A[(int64_t)(k + j) * n + i] : make_double2(0.0, 0.0);
    }
#pragma unroll
    for (int cc = 0; cc < kLuPanel; ++cc) {
      if (cc >= w) break;
      double2 v[R];
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const int i = row0 + tid + q * kLuRows;
        v[q] = i < N ? C[cc * n + i] : make_double2(0.0, 0.0);
      }
      // (the products are summed first: one rounding of C per panel, not one per column)
      double2 s[R];
#pragma unroll
      for (int q = 0; q < R; ++q) s[q] = make_double2(0.0, 0.0);
#pragma unroll
      for (int j = 0; j < kLuPanel; ++j) {
        const double2 u = us[j][cc];
#pragma unroll
        for (int q = 0; q < R; ++q) s[q] = cfma(s[q], l[q][j], u);
      }
#pragma unroll
      for (int q = 0; q < R; ++q) v[q] = make_double2(v[q].x - s[q].x, v[q].y - s[q].y);
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const int i = row0 + tid + q * kLuRows;
        if (i < N) C[cc * n + i] = v[q];
      }
    }
    if (strip != sk + 1) return;
    __syncthreads();
  }
  // factor the strip: row row0 + tid + q kLuRows in a[q] (row0 = c0; written above by this thread)
  double2 a[R][kLuPanel];
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const int i = row0 + tid + q * kLuRows;
#pragma unroll
    for (int cc = 0; cc < kLuPanel; ++cc) a[q][cc] = cc < w && i < N ? C[cc * n + i] : make_double2(0.0, 0.0);
    if (i < N) {
      const int o = k >= 0 ? origin[i] : i;
      origin_out[i] = o;
#pragma unroll
      for (int cc = 0; cc < kLuPanel; ++cc)
        if (cc < w && o == c0 + cc) a[q][cc].x += 1.0;
    }
  }
#pragma unroll
  for (int j = 0; j < kLuPanel; ++j) {
    if (j >= w) break;
    // pivot: the largest |re| + |im| of the rows from j on, the first of equals (no row but NaN: j)
    constexpr unsigned kNone = 0xffffffffu;
    unsigned long long key = 0;
    int best = -1;  // the lane's q
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int i = tid + q * kLuRows;
      const double v = fabs(a[q][j].x) + fabs(a[q][j].y);
      const unsigned long long kq = (unsigned long long)__double_as_longlong(v);
      if (i >= j && row0 + i < N && v >= 0.0 && (best < 0 || kq > key)) {
        key = kq;
        best = q;
      }
    }
    const unsigned long long most = max_xor(max_xor(max_row(key), 16), 32);
    unsigned index = kNone;
#pragma unroll
    for (int q = R - 1; q >= 0; --q) {
      const unsigned long long lanes = __ballot(best == q && key == most);
      if (lanes) index = (unsigned)((tid & ~63) + q * kLuRows + __ffsll((long long)lanes) - 1);
    }
    if ((tid & 63) == 0) {
      redk[tid >> 6] = most;
      redi[tid >> 6] = index;
    }
    __syncthreads();
    const unsigned long long wave_key = redk[tid & (kLuWaves - 1)];
    const unsigned wave_index = redi[tid & (kLuWaves - 1)];
    // (a wave without rows has the key 0 and no index)
    const unsigned first = min_row(wave_key == max_row(wave_key) ? wave_index : kNone);
    const int at = first == kNone ? j : (int)first;
#pragma unroll
    for (int q = 0; q < R; ++q)
      if (tid + q * kLuRows == at) {
#pragma unroll
        for (int cc = 0; cc < kLuPanel; ++cc) prow[cc] = a[q][cc];
      }
    if (tid == j) {
#pragma unroll
      for (int cc = 0; cc < kLuPanel; ++cc) orow[cc] = a[0][cc];
      pivots[j] = row0 + at;
      ipiv[c0 + j] = row0 + at + 1;
    }
    __syncthreads();
    if (at != j) {
      if (tid == j) {
#pragma unroll
        for (int cc = 0; cc < kLuPanel; ++cc) a[0][cc] = prow[cc];
      }
#pragma unroll
      for (int q = 0; q < R; ++q)
        if (tid + q * kLuRows == at) {
#pragma unroll
          for (int cc = 0; cc < kLuPanel; ++cc) a[q][cc] = orow[cc];
        }
    }
    // 1 / pivot, scaled by a power of two (a zero pivot is reported and leaves its column)
    const double2 p = prow[j];
    const bool zero = p.x == 0.0 && p.y == 0.0;
    if (zero && tid == 0 && *info == 0) *info = c0 + j + 1;
    const int e = zero ? 0 : -ilogb(fmax(fabs(p.x), fabs(p.y)));
    const double px = ldexp(p.x, e), py = ldexp(p.y, e);
    const double d = zero ? 0.0 : 1.0 / (px * px + py * py);
    const double ix = ldexp(px * d, e), iy = -ldexp(py * d, e);
#pragma unroll
    for (int q = 0; q < R; ++q) {
      if (tid + q * kLuRows <= j) continue;
      const double2 v = a[q][j];
      const double2 lv = make_double2(v.x * ix - v.y * iy, v.x * iy + v.y * ix);
      a[q][j] = lv;
#pragma unroll
      for (int cc = j + 1; cc < kLuPanel; ++cc) a[q][cc] = csub(a[q][cc], lv, prow[cc]);
    }
  }
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const int i = row0 + tid + q * kLuRows;
#pragma unroll
    for (int cc = 0; cc < kLuPanel; ++cc)
      if (cc < w && i < N) C[cc * n + i] = a[q][cc];
  }
  if (tid < 64) {
    // the exchanges as one permutation: lane t holds row[t] and src[t]
    int count = w, row = tid < w ? c0 + tid : -1, src = tid;
    for (int j = 0; j < w; ++j) {
      const int pj = pivots[j];
      const unsigned long long there = __ballot(row == pj);
      int b = count;
      if (there) {
        b = __ffsll((long long)there) - 1;
      } else {
        if (tid == count) row = pj;
        ++count;
      }
      const int sj = __shfl(src, j), sb = __shfl(src, b);
      if (tid == j) src = sb;
      if (tid == b) src = sj;
    }
    const int from = __shfl(row, src);
    LuPerm& pm = perms[strip];
    if (tid < count) {
      pm.row[tid] = row;
      pm.src[tid] = src;
      pm.origin[tid] = k >= 0 ? origin[from] : from;
    }
    if (tid == 0) pm.count = count;
  }
}

// Factors I + A. ipiv [n], info [1], perms [strips] and origin [2 n] on the
// device; info is the first zero pivot's column (1-based), or 0
void lu_factor(double2* A, int64_t n, int* ipiv, int* info, LuPerm* perms, int* origin, hipStream_t s) {
  const int strips = (int)((n + kLuPanel - 1) / kLuPanel);
  (void)hipMemsetAsync(info, 0, sizeof(int), s);
  for (int st = -1; st < strips; ++st) {
    const int k = st * kLuPanel;
    const int blocks = st < 0 ? 1 : strips - 1;  // all strips but the factored one
    if (blocks == 0) break;
    const auto kern = n - (k + kLuPanel) > kLuRows ? lu_step_kernel<2> : lu_step_kernel<1>;
    hipLaunchKernelGGL(kern, dim3(blocks), dim3(kLuRows), 0, s, A, n, k, perms, (const int*)origin + (st & 1) * n,
                       origin + ((st + 1) & 1) * n, ipiv, info);
  }
}

}  // namespace

namespace smh {

void lu_release(smh_op* op) {
  if (op->d_lu) (void)hipFree(op->d_lu);
  if (op->d_piv) (void)hipFree(op->d_piv);
  if (op->blas) (void)rocblas_destroy_handle((rocblas_handle)op->blas);
  op->d_lu = nullptr;
  op->d_piv = nullptr;
  op->blas = nullptr;
  op->lu_t.clear();
}

int lu_solve(smh_op* op, const double* t_diag, const double* rhs, double* x, int64_t nrhs, double* stats) {
  smh_ctx* ctx = op->ctx;
  SMH_CHECK(ctx, op->kind == 2 && op->d_W64, SMH_ERR_UNSUPPORTED,
            "LU factorization needs the stored (explicit) coupling matrix");
  const auto t0 = std::chrono::steady_clock::now();
  hipStream_t s = ctx->stream;
  const int64_t n = op->n_part * op->B;
  SMH_CHECK(ctx, n < (int64_t)1 << 31 && n * n < (int64_t)1 << 62, SMH_ERR_ARG, "matrix too large");
  if (!op->blas) {
    rocblas_handle h = nullptr;
    SMH_CHECK(ctx, rocblas_create_handle(&h) == rocblas_status_success, SMH_ERR_HIP, "rocblas_create_handle failed");
    op->blas = h;
  }
  rocblas_handle h = (rocblas_handle)op->blas;
  SMH_CHECK(ctx, rocblas_set_stream(h, s) == rocblas_status_success, SMH_ERR_HIP, "rocblas_set_stream failed");
  int rc = op_reserve_packed(op, nrhs);
  if (rc) return rc;
  double2 *d_t = nullptr, *d_b = nullptr, *d_x = nullptr, *d_y = nullptr;
  double* d_parts = nullptr;
  int* d_info = nullptr;
  LuPerm* d_perms = nullptr;
  int* d_origin = nullptr;
  constexpr int kParts = 256;
  auto done = [&](int code) {
    void* p[] = {d_t, d_b, d_x, d_y, d_parts, d_info, d_perms, d_origin};
    for (void* q : p)
      if (q) (void)hipFree(q);
    return code;
  };
  if (hipMalloc(&d_t, n * sizeof(double2)) != hipSuccess || hipMalloc(&d_b, nrhs * n * sizeof(double2)) != hipSuccess ||
      hipMalloc(&d_x, nrhs * n * sizeof(double2)) != hipSuccess ||
      hipMalloc(&d_y, nrhs * n * sizeof(double2)) != hipSuccess ||
      hipMalloc(&d_parts, nrhs * kParts * 2 * sizeof(double)) != hipSuccess ||
      hipMalloc(&d_info, sizeof(int)) != hipSuccess)
    return done(smh_fail(ctx, SMH_ERR_HIP, "device allocation failed (LU solve vectors)"));
#define LU_HIP(call)                                                                                           \
  do {                                                                                                         \
    hipError_t e__ = (call);                                                                                   \
    if (e__ != hipSuccess)                                                                                     \
      return done(smh_fail(ctx, SMH_ERR_HIP, "%s failed: %s (%s:%d)", #call, hipGetErrorString(e__), __FILE__, \
                           __LINE__));                                                                         \
  } while (0)
#define LU_TRY(call)         \
  do {                       \
    int rc__ = (call);       \
    if (rc__) return done(rc__); \
  } while (0)
  LU_HIP(hipMemcpyAsync(op->d_pk_in, t_diag, op->n_unk * sizeof(double2), hipMemcpyDefault, s));
  LU_TRY(op_unpack(op, SMH_FP64, op->d_pk_in, d_t));
  // the factors of an earlier call serve while T is the same (the reference
  // keeps LU_piv on the master matrix)
  const std::vector<double> tkey(t_diag, t_diag + 2 * op->n_unk);
  if (!op->d_lu || op->lu_t != tkey) {
    if (!op->d_lu) {
      LU_HIP(hipMalloc(&op->d_lu, (size_t)n * n * sizeof(double2)));
      LU_HIP(hipMalloc(&op->d_piv, (size_t)n * sizeof(int)));
    }
    op->lu_t.clear();
    const bool own = n <= 2 * kLuRows;
    hipLaunchKernelGGL(master_dense_kernel, dim3(blocks_of(n * n)), dim3(256), 0, s, (const double2*)op->d_W64,
                       (const double2*)d_t, n, own ? 0.0 : 1.0, op->d_lu);
    LU_HIP(hipGetLastError());
    if (own) {
      LU_HIP(hipMalloc(&d_perms, (size_t)((n + kLuPanel - 1) / kLuPanel) * sizeof(LuPerm)));
      LU_HIP(hipMalloc(&d_origin, (size_t)2 * n * sizeof(int)));
      lu_factor(op->d_lu, n, op->d_piv, d_info, d_perms, d_origin, s);
      LU_HIP(hipGetLastError());
    } else {
      const rocblas_status st = rocsolver_zgetrf(h, (rocblas_int)n, (rocblas_int)n,
                                                 reinterpret_cast<rocblas_double_complex*>(op->d_lu), (rocblas_int)n,
                                                 op->d_piv, d_info);
      if (st != rocblas_status_success)
        return done(smh_fail(ctx, SMH_ERR_HIP, "rocsolver_zgetrf failed (%d)", (int)st));
    }
    int info = 0;
    LU_HIP(hipMemcpyAsync(&info, d_info, sizeof(int), hipMemcpyDeviceToHost, s));
    LU_HIP(hipStreamSynchronize(s));
    if (info != 0)
      return done(smh_fail(ctx, SMH_ERR_ARG, "the master matrix is singular (zero pivot %d of %lld)", info,
                           (long long)n));
    op->lu_t = tkey;
  }
  // right-hand sides in the padded layout, one column each
  LU_HIP(hipMemcpyAsync(op->d_pk_in, rhs, (size_t)nrhs * op->n_unk * sizeof(double2), hipMemcpyDefault, s));
  for (int64_t r = 0; r < nrhs; ++r) {
    LU_TRY(op_unpack(op, SMH_FP64, op->d_pk_in + r * op->n_unk, d_b + r * n));
  }
  LU_HIP(hipMemcpyAsync(d_x, d_b, (size_t)nrhs * n * sizeof(double2), hipMemcpyDeviceToDevice, s));
  const rocblas_status st = rocsolver_zgetrs(h, rocblas_operation_transpose, (rocblas_int)n, (rocblas_int)nrhs,
                                             reinterpret_cast<rocblas_double_complex*>(op->d_lu), (rocblas_int)n,
                                             op->d_piv, reinterpret_cast<rocblas_double_complex*>(d_x),
                                             (rocblas_int)n);
  if (st != rocblas_status_success) return done(smh_fail(ctx, SMH_ERR_HIP, "rocsolver_zgetrs failed (%d)", (int)st));
  // certificate: FP64 residual of every solution
  for (int64_t r = 0; r < nrhs; ++r) LU_TRY(explicit_apply(op, SMH_FP64, d_x + r * n, d_y + r * n, false));
  hipLaunchKernelGGL(residual_parts_kernel, dim3(kParts, (unsigned)nrhs), dim3(256), 0, s, (const double2*)d_b,
                     (const double2*)d_x, (const double2*)d_y, (const double2*)d_t, n, d_parts);
  LU_HIP(hipGetLastError());
  std::vector<double> parts((size_t)nrhs * kParts * 2);
  LU_HIP(hipMemcpyAsync(parts.data(), d_parts, parts.size() * sizeof(double), hipMemcpyDeviceToHost, s));
  for (int64_t r = 0; r < nrhs; ++r) LU_TRY(op_pack(op, SMH_FP64, d_x + r * n, op->d_pk_out + r * op->n_unk));
  LU_HIP(hipMemcpyAsync(x, op->d_pk_out, (size_t)nrhs * op->n_unk * sizeof(double2), hipMemcpyDefault, s));
  LU_HIP(hipStreamSynchronize(s));
  double worst = 0;
  for (int64_t r = 0; r < nrhs; ++r) {
    double rr = 0, bb = 0;
    for (int k = 0; k < kParts; ++k) {
      rr += parts[((size_t)r * kParts + k) * 2];
      bb += parts[((size_t)r * kParts + k) * 2 + 1];
    }
    worst = std::max(worst, bb > 0 ? std::sqrt(rr / bb) : 0.0);
  }
  if (stats) {
    for (int k = 0; k < 8; ++k) stats[k] = 0;
    stats[1] = (double)nrhs;  // FP64 matvecs (the residual certificates)
    stats[3] = worst;
    stats[4] = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  }
#undef LU_HIP
#undef LU_TRY
  return done(SMH_OK);
}

}  // namespace smh
