// GMRES for (1 - T W) b = T a on the GPU.
//
// Vectors live on the device in the padded layout [n_part][B] (complex FP64);
// slots a particle does not have carry T = 0 and stay zero. Arnoldi uses
// classical Gram-Schmidt applied twice (CGS2) in FP64 with fused multi-dot
// and multi-axpy kernels.
//
// One driver for KB = 1 right-hand side (single right-hand sides, operators
// without the kBatch-RHS kernels) and for KB = kBatch right-hand sides at a
// time over every ensemble ("segment") of the operator: every (segment,
// right-hand side) pair is a system of its own (its own Arnoldi scalars, Givens
// rotations and convergence), all systems share each coupling matvec launch,
// and the Givens rotations, the back-substitution and the restart bookkeeping
// run on the device. One Arnoldi step (matvec, CGS2, norm, rotation,
// normalisation) is a fixed launch sequence that is captured once per (step,
// precision, preconditioner) in a hipGraph and replayed; the last kernel of a
// step writes the count of still-active systems to pinned host memory, the one
// value the host waits for. With a right block preconditioner P (op->d_P) the
// steps apply M P and the update is x += P V y.
//
// SMH_SOLVE_FP64: restarted GMRES with FP64 coupling matvecs, x0 = rhs and
//   stopping rule ||rhs - M x|| <= tol ||rhs|| (smuthi's scipy call,
//   linear_system.py:285-286).
// SMH_SOLVE_MIXED: FP64 iterative refinement from x = 0: an inner GMRES with
//   FP32 coupling matvecs (FP64 Arnoldi) solves M d = r to
//   max(tol/2 ||rhs||, kInnerRel ||r||), x += d, r = rhs - M x with the FP64
//   matvec, until the FP64 residual meets tol. kInnerRel sits at the FP32
//   operator's resolution, so for tolerances down to ~1e-6 the first sweep
//   usually suffices and one FP64 matvec checks it. Inner solves run one
//   restart cycle per sweep, so the FP64 residual is taken after every cycle
//   (a reduced-precision operator never restarts on its own residuals).
// SMH_SOLVE_MIXED16: the same refinement with FP16-operand matvecs in the
//   inner GMRES (batched radial solves), whose target kInnerRel16 sits at
//   that operator's resolution (a few 1e-4): each sweep gains about three
//   digits, so tolerances near 1e-6 take two sweeps. Between sweeps the
//   residual comes from the FP32 matvec; the FP64 residual certifies the
//   result once that meets the tolerance.
#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdlib>
#include <map>
#include <set>

#include "smh_op.h"

namespace {

int blocks_for(int64_t n, int t = 256) { return (int)((n + t - 1) / t); }

constexpr int kDotThreads = 256;
constexpr int kDotBlocks = 512;
constexpr int kMaxBasis = 128;
constexpr double kInnerRel = 2e-7;    // inner (FP32-matvec) GMRES target relative to the current FP64 residual
constexpr double kInnerRel16 = 1e-3;  // the same for FP16-operand matvecs
// FP32 residuals drive FP16 sweeps while above this fraction of ||b|| (about
// 30 times the FP32 matvec's error)
constexpr double kFp32ResidualFloor = 1e-5;

__global__ void to_fp32_kernel(const double2* __restrict__ v, float2* out, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = make_float2((float)v[i].x, (float)v[i].y);
}

__global__ void sub_kernel(const double2* __restrict__ a, const double2* __restrict__ b, double2* out, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = make_double2(a[i].x - b[i].x, a[i].y - b[i].y);
}

__global__ void add_kernel(double2* a, const double2* __restrict__ b, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) a[i] = make_double2(a[i].x + b[i].x, a[i].y + b[i].y);
}

__global__ void zero2_kernel(double2* p, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    p[i] = make_double2(0.0, 0.0);
}
__global__ void zero_int_kernel(int* p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}
__global__ void zero_f2_kernel(float2* p, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    p[i] = make_float2(0.f, 0.f);
}

// ---------------------------------------------------------------------------
// KB right-hand sides x segments: element e = (particle * B + n) * KB + r of a
// padded vector; system sys = segment(particle) * KB + r
// ---------------------------------------------------------------------------
constexpr int kB = smh::kBatchRhs;

// partial[((s * nblk + b) * kMaxBasis + j) * KB + r]: block b's share of
// conj(V_j) . w over segment s and right-hand side r (grid: nblk x n_seg; a
// thread sees one r, since segments start at multiples of KB elements and
// the block stride is a multiple of KB)
template <int KB>
__global__ void __launch_bounds__(kDotThreads) sdot_kernel(const double2* __restrict__ V, int64_t ld, int nv,
                                                           const double2* __restrict__ w, int64_t per_part,
                                                           const int64_t* __restrict__ seg_off, double2* partial) {
  __shared__ double2 red[kDotThreads];
  const int s = blockIdx.y, b = blockIdx.x, nblk = gridDim.x;
  const int64_t e0 = seg_off[s] * per_part, e1 = seg_off[s + 1] * per_part;
  for (int j = 0; j < nv; ++j) {
    const double2* v = V + (size_t)j * ld;
    double re = 0, im = 0;
    for (int64_t e = e0 + (int64_t)b * blockDim.x + threadIdx.x; e < e1; e += (int64_t)nblk * blockDim.x) {
      const double2 a = v[e], c = w[e];
      re += a.x * c.x + a.y * c.y;
      im += a.x * c.y - a.y * c.x;
    }
    red[threadIdx.x] = make_double2(re, im);
    __syncthreads();
    for (int st = blockDim.x / 2; st >= KB; st >>= 1) {  // strides keep e % KB
      if ((int)threadIdx.x < st) {
        red[threadIdx.x].x += red[threadIdx.x + st].x;
        red[threadIdx.x].y += red[threadIdx.x + st].y;
      }
      __syncthreads();
    }
    if ((int)threadIdx.x < KB)
      partial[(((size_t)s * nblk + b) * kMaxBasis + j) * KB + threadIdx.x] = red[threadIdx.x];
    __syncthreads();
  }
}

// out[(s * KB + r) * ldo + j] = sum over the nblk partials, fixed-order tree;
// one workgroup per (j, r) and segment
template <int KB>
__global__ void __launch_bounds__(256) sreduce_kernel(const double2* __restrict__ partial, int nblk, double2* out,
                                                      int ldo) {
  const int j = blockIdx.x / KB, r = blockIdx.x % KB, s = blockIdx.y;
  __shared__ double2 red[256];
  double re = 0, im = 0;
  for (int b = threadIdx.x; b < nblk; b += blockDim.x) {
    const double2 p = partial[(((size_t)s * nblk + b) * kMaxBasis + j) * KB + r];
    re += p.x;
    im += p.y;
  }
  red[threadIdx.x] = make_double2(re, im);
  __syncthreads();
  for (int w = blockDim.x / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) {
      red[threadIdx.x].x += red[threadIdx.x + w].x;
      red[threadIdx.x].y += red[threadIdx.x + w].y;
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) out[((size_t)s * KB + r) * ldo + j] = red[0];
}

template <int KB>
__device__ inline int sys_of(int64_t e, int64_t per_part, const int* __restrict__ seg_of) {
  const int r = (int)(e % KB);
  return (seg_of ? seg_of[e / per_part] : 0) * KB + r;
}

// w[e] += sgn * sum_j V_j[e] c[sys(e) * ldc + j]
template <int KB>
__global__ void saxpy_kernel(const double2* __restrict__ V, int64_t ld, int nv, const double2* __restrict__ c,
                             int ldc, double sgn, double2* w, int64_t n8, int64_t per_part,
                             const int* __restrict__ seg_of) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n8) return;
  const double2* cs = c + (size_t)sys_of<KB>(e, per_part, seg_of) * ldc;
  double2 acc = w[e];
  for (int j = 0; j < nv; ++j) {
    const double2 v = V[(size_t)j * ld + e], cj = cs[j];
    acc.x += sgn * (v.x * cj.x - v.y * cj.y);
    acc.y += sgn * (v.x * cj.y + v.y * cj.x);
  }
  w[e] = acc;
}

// dst = src sc[sys]; with `live` the launch also hands the host that count
// (pinned memory; the kernel that wrote it has ended)
template <int KB>
__global__ void sscale_kernel(const double2* __restrict__ src, const double* __restrict__ sc, double2* dst,
                              int64_t n8, int64_t per_part, const int* __restrict__ seg_of, const int* live,
                              int* host_live) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (live && e == 0) *host_live = *live;
  if (e >= n8) return;
  const double f = sc[sys_of<KB>(e, per_part, seg_of)];
  dst[e] = make_double2(src[e].x * f, src[e].y * f);
}

// out = v - t o y with t per unknown, shared by the right-hand sides (master
// matrix 1 - T W applied after the coupling matvec)
template <int KB>
__global__ void bmaster_fp64_kernel(const double2* __restrict__ v, const double2* __restrict__ t,
                                    const double2* __restrict__ y, double2* out, int64_t n8) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n8) return;
  const double2 a = t[e / KB], b = y[e];
  out[e] = make_double2(v[e].x - (a.x * b.x - a.y * b.y), v[e].y - (a.x * b.y + a.y * b.x));
}

// FP64 padded [n][kB] -> FP32 input of the batched kernel (b32_index layout)
__global__ void to_fp32_b32_kernel(const double2* __restrict__ v, float2* out, int64_t n8, int B, int S,
                                   const int* __restrict__ slot) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n8) return;
  const int r = (int)(e % kB);
  const int64_t ip = e / kB, p = ip / B;
  out[smh::b32_index(p, (int)(ip - p * B), r, S, slot)] = make_float2((float)v[e].x, (float)v[e].y);
}

template <int KB>
__global__ void bmaster_fp32_kernel(const double2* __restrict__ v, const double2* __restrict__ t,
                                    const float2* __restrict__ y, double2* out, int64_t n8) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n8) return;
  const double2 a = t[e / KB];
  const double bx = y[e].x, by = y[e].y;
  out[e] = make_double2(v[e].x - (a.x * bx - a.y * by), v[e].y - (a.x * by + a.y * bx));
}

__device__ inline double2 cmul2(double2 a, double2 b) { return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x); }
__device__ inline double2 cconj2(double2 a) { return make_double2(a.x, -a.y); }
__device__ inline double2 cdiv2(double2 a, double2 b) {
  const double d = b.x * b.x + b.y * b.y;
  return make_double2((a.x * b.x + a.y * b.y) / d, (a.y * b.x - a.x * b.y) / d);
}

// Start of a restart cycle (one thread per system): beta = ||r|| from the norm
// dot, the system runs this cycle if active, beta > atol and it has steps left;
// nlive[restart] counts the systems that run.
__global__ void cycle_init_kernel(const double2* __restrict__ nrm, const double* __restrict__ atol,
                                  const int* __restrict__ active, const int* __restrict__ left, int nsys, int restart, double2* g, int* live,
                                  double* scale, double* res, int* kr, int* nlive) {
  const int sys = blockIdx.x * blockDim.x + threadIdx.x;
  if (sys >= nsys) return;
  const double beta = sqrt(fmax(0.0, nrm[sys].x));
  res[sys] = beta;
  const bool c = active[sys] && beta > atol[sys] && beta > 0.0 && left[sys] > 0;
  live[sys] = c ? 1 : 0;
  kr[sys] = 0;
  scale[sys] = c ? 1.0 / beta : 0.0;
  double2* gs = g + (size_t)sys * (restart + 1);
  for (int j = 0; j <= restart; ++j) gs[j] = make_double2(0.0, 0.0);
  gs[0] = make_double2(c ? beta : 0.0, 0.0);
  if (c) atomicAdd(&nlive[restart], 1);
}

// Arnoldi step k of one live system: the new Hessenberg column col[0..k] (the
// sum of the two CGS passes) with h_{k+1,k} = hn = ||w||, the previous Givens
// rotations applied to it, a new rotation zeroing h_{k+1,k} and the rotated
// right-hand side g. Returns whether the system goes on: it stops when its
// least-squares residual |g_{k+1}| reaches atol.
__device__ inline bool givens_step(int k, double2* col, double hn, double atol, int restart, double2* Hs,
                                   double2* css, double2* sns, double2* gs) {
  double2 a = col[0];
  for (int j = 0; j < k; ++j) {
    const double2 b = col[j + 1];
    const double2 c = css[j], s = sns[j];
    const double2 u = cmul2(cconj2(c), a), v = cmul2(cconj2(s), b);
    const double2 p = cmul2(s, a), q = cmul2(c, b);
    Hs[(size_t)j * restart + k] = make_double2(u.x + v.x, u.y + v.y);
    a = make_double2(q.x - p.x, q.y - p.y);
  }
  const double den = sqrt(a.x * a.x + a.y * a.y + hn * hn);
  const double2 c = den > 0 ? make_double2(a.x / den, a.y / den) : make_double2(1.0, 0.0);
  const double2 s = den > 0 ? make_double2(hn / den, 0.0) : make_double2(0.0, 0.0);
  const double2 u = cmul2(cconj2(c), a);
  Hs[(size_t)k * restart + k] = make_double2(u.x + s.x * hn, u.y - s.y * hn);
  const double2 gk = gs[k];
  const double2 gn = cmul2(s, gk);
  gs[k + 1] = make_double2(-gn.x, -gn.y);
  gs[k] = cmul2(cconj2(c), gk);
  css[k] = c;
  sns[k] = s;
  const double gr = sqrt(gn.x * gn.x + gn.y * gn.y);
  return !(gr <= atol || hn == 0.0);
}

// The step's rotations (one thread per system) and the normalisation of w;
// nlive[k] counts the systems still running after this step (no more than left
// steps of the cycle).
__global__ void givens_kernel(int k, double2* h1, const double2* __restrict__ h2, int ldh,
                              const double2* __restrict__ hn2, const double* __restrict__ atol,
                              const int* __restrict__ left, int nsys, int restart,
                              int* live, double2* H, double2* cs, double2* sn, double2* g, int* kr, double* scale,
                              int* nlive) {
  const int sys = blockIdx.x * blockDim.x + threadIdx.x;
  if (sys >= nsys) return;
  if (!live[sys]) {
    scale[sys] = 0.0;
    return;
  }
  const double hn = sqrt(fmax(0.0, hn2[sys].x));
  double2* col = h1 + (size_t)sys * ldh;
  for (int j = 0; j <= k; ++j) {
    const double2 a = col[j], b = h2[(size_t)sys * ldh + j];
    col[j] = make_double2(a.x + b.x, a.y + b.y);
  }
  const bool on = givens_step(k, col, hn, atol[sys], restart, H + (size_t)sys * (restart + 1) * restart,
                              cs + (size_t)sys * restart, sn + (size_t)sys * restart, g + (size_t)sys * (restart + 1)) &&
                  k + 1 < left[sys];
  kr[sys] = k + 1;
  scale[sys] = hn > 0 ? 1.0 / hn : 0.0;
  if (!on)
    live[sys] = 0;
  else
    atomicAdd(&nlive[k], 1);
}

// Everything of an Arnoldi step that follows the matvec, for one system whose
// vector fits a workgroup's registers (kSmallVector entries): CGS2 against
// V_0..V_k, the norm, the rotations and V_{k+1}. Bound by its dependent passes
// over V, which one CU reads from its XCD's L2 (4 MB): beyond kSmallBasis
// entries of basis the launches it replaces (two dots, two reductions, two
// updates, norm, rotation, scaling), which spread them over the chip, are the
// faster ones. A whole step of 4092 unknowns: 81 us against 100 below k = 4, 237
// against 265 below k = 48, 300 against 333 below 64, but 536 against 437 from k
// = 64 to 96; of 2100 unknowns 61 against 71 below k = 4, 429 against 450 below
// k = 126; of 600 unknowns 45 against 60 and 336 against 406.
constexpr int kSmallThreads = 1024, kSmallPer = 4, kSmallVector = kSmallThreads * kSmallPer;
constexpr int64_t kSmallBasis = (int64_t)1 << 18;
__global__ void __launch_bounds__(kSmallThreads)
    arnoldi_small_kernel(int k, double2* V, const double2* __restrict__ wv, int n, const double* __restrict__ atol,
                         const int* __restrict__ left, int restart, int* live, double2* H, double2* cs, double2* sn, double2* g, int* kr,
                         int* nlive, int* host_live) {
  __shared__ double2 red[kSmallThreads / 64][kMaxBasis + 1];
  __shared__ double2 h[kMaxBasis + 1], col[kMaxBasis + 1], css[kMaxBasis], sns[kMaxBasis];
  __shared__ double scale;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  double2 w[kSmallPer];
#pragma unroll
  for (int u = 0; u < kSmallPer; ++u) {
    const int e = u * kSmallThreads + tid;
    w[u] = e < n ? wv[e] : make_double2(0.0, 0.0);
  }
  if (tid < k) {
    css[tid] = cs[tid];
    sns[tid] = sn[tid];
  }
  // sum of (re, im) over the wave into red[wave][j]
  auto wave_sum = [&](int j, double re, double im) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      re += __shfl_xor(re, off);
      im += __shfl_xor(im, off);
    }
    if (lane == 0) red[wave][j] = make_double2(re, im);
  };
  auto block_sum = [&](int nv) {
    __syncthreads();
    if (tid < nv) {
      double2 s = red[0][tid];
      for (int q = 1; q < kSmallThreads / 64; ++q) {
        s.x += red[q][tid].x;
        s.y += red[q][tid].y;
      }
      h[tid] = s;
    }
    __syncthreads();
  };
  for (int pass = 0; pass < 2; ++pass) {
#pragma unroll 2
    for (int j = 0; j <= k; ++j) {
      double re = 0, im = 0;
#pragma unroll
      for (int u = 0; u < kSmallPer; ++u) {
        const int e = u * kSmallThreads + tid;
        if (e < n) {
          const double2 a = V[(size_t)j * n + e];
          re += a.x * w[u].x + a.y * w[u].y;
          im += a.x * w[u].y - a.y * w[u].x;
        }
      }
      wave_sum(j, re, im);
    }
    block_sum(k + 1);
    if (tid <= k) {
      if (pass == 0)
        col[tid] = h[tid];
      else
        col[tid] = make_double2(col[tid].x + h[tid].x, col[tid].y + h[tid].y);
    }
#pragma unroll 4
    for (int j = 0; j <= k; ++j) {
      const double2 c = h[j];
#pragma unroll
      for (int u = 0; u < kSmallPer; ++u) {
        const int e = u * kSmallThreads + tid;
        if (e < n) {
          const double2 v = V[(size_t)j * n + e];
          w[u].x -= v.x * c.x - v.y * c.y;
          w[u].y -= v.x * c.y + v.y * c.x;
        }
      }
    }
    __syncthreads();  // h is read by all before the next sums
  }
  double nn = 0;
#pragma unroll
  for (int u = 0; u < kSmallPer; ++u) nn += w[u].x * w[u].x + w[u].y * w[u].y;
  wave_sum(0, nn, 0.0);
  block_sum(1);
  if (tid == 0) {
    double f = 0.0;
    if (live[0]) {
      const double hn = sqrt(fmax(0.0, h[0].x));
      const bool on = givens_step(k, col, hn, atol[0], restart, H, css, sns, g) && k + 1 < left[0];
      cs[k] = css[k];
      sn[k] = sns[k];
      kr[0] = k + 1;
      f = hn > 0 ? 1.0 / hn : 0.0;
      if (!on) live[0] = 0;
      nlive[k] = on ? 1 : 0;
      *host_live = on ? 1 : 0;
    } else {
      *host_live = nlive[k];
    }
    scale = f;
  }
  __syncthreads();
  const double f = scale;
#pragma unroll
  for (int u = 0; u < kSmallPer; ++u) {
    const int e = u * kSmallThreads + tid;
    if (e < n) V[(size_t)(k + 1) * n + e] = make_double2(w[u].x * f, w[u].y * f);
  }
}

// End of a cycle (one thread per system): y = R^{-1} g over the system's
// kr steps (zero beyond), and its least-squares residual estimate |g_kr|. The
// cycle's steps come off the system's steps left: `used` of them, or (used < 0)
// its own.
__global__ void backsub_kernel(int nsys, int restart, const double2* __restrict__ H, const double2* __restrict__ g,
                               const int* __restrict__ kr, double2* yv, int ldy, double* res, int used, int* left) {
  const int sys = blockIdx.x * blockDim.x + threadIdx.x;
  if (sys >= nsys) return;
  const int m = kr[sys];
  left[sys] -= used >= 0 ? used : m;
  const double2* Hs = H + (size_t)sys * (restart + 1) * restart;
  const double2* gs = g + (size_t)sys * (restart + 1);
  double2* y = yv + (size_t)sys * ldy;
  for (int j = 0; j < ldy; ++j) y[j] = make_double2(0.0, 0.0);
  for (int i = m - 1; i >= 0; --i) {
    double2 sum = gs[i];
    for (int j = i + 1; j < m; ++j) {
      const double2 p = cmul2(Hs[(size_t)i * restart + j], y[j]);
      sum.x -= p.x;
      sum.y -= p.y;
    }
    y[i] = cdiv2(sum, Hs[(size_t)i * restart + i]);
  }
  if (m > 0) res[sys] = sqrt(gs[m].x * gs[m].x + gs[m].y * gs[m].y);
}

// y_i = sum_k P[i][k] x_{nbr[i][k]} (+ y_i) for kB padded vectors: one
// workgroup per particle, thread (n1, r), the emitter's vector staged in LDS
__global__ void __launch_bounds__(256) precond_kernel(const double2* __restrict__ P, const int* __restrict__ nbr,
                                                      int k1, const double2* __restrict__ x, double2* y, int B,
                                                      int accumulate) {
  extern __shared__ double2 xs[];  // [B][kB]
  const int64_t p = blockIdx.x;
  const int nel = B * kB;
  double2 acc[2] = {make_double2(0.0, 0.0), make_double2(0.0, 0.0)};
  for (int k = 0; k < k1; ++k) {
    const int j = nbr[p * k1 + k];
    if (j < 0) continue;
    __syncthreads();
    const double2* xj = x + (size_t)j * nel;
    for (int e = threadIdx.x; e < nel; e += blockDim.x) xs[e] = xj[e];
    __syncthreads();
    const double2* Pk = P + ((size_t)p * k1 + k) * B * B;
    for (int u = 0; u < 2; ++u) {
      const int t = threadIdx.x + u * blockDim.x;
      if (t >= nel) break;
      const int n1 = t / kB, r = t - n1 * kB;
      double re = acc[u].x, im = acc[u].y;
      for (int n2 = 0; n2 < B; ++n2) {
        const double2 a = Pk[(size_t)n1 * B + n2], b = xs[n2 * kB + r];
        re += a.x * b.x - a.y * b.y;
        im += a.x * b.y + a.y * b.x;
      }
      acc[u] = make_double2(re, im);
    }
  }
  for (int u = 0; u < 2; ++u) {
    const int t = threadIdx.x + u * blockDim.x;
    if (t >= nel) break;
    double2* out = y + (size_t)p * nel + t;
    double re = acc[u].x, im = acc[u].y;
    if (accumulate) {
      re += out->x;
      im += out->y;
    }
    *out = make_double2(re, im);
  }
}

// ---- per-operator workspace ------------------------------------------------
// One set of vectors and scalars per KB (single and batched systems).
struct SolveWs {
  int64_t n8 = 0;
  int restart = 0, nsys = 0, nblk = 0;
  double2 *V = nullptr, *w = nullptr, *t = nullptr, *partial = nullptr, *h1 = nullptr, *h2 = nullptr,
          *hn = nullptr, *H = nullptr, *cs = nullptr, *sn = nullptr, *g = nullptr, *yv = nullptr, *y64 = nullptr,
          *b = nullptr, *x = nullptr, *d = nullptr, *r = nullptr, *pv = nullptr, *tmp = nullptr;
  // atol, res, left and active are one block: uploaded, and the middle two read back, in one copy
  double *atol = nullptr, *scale = nullptr, *res = nullptr;
  int *live = nullptr, *kr = nullptr, *nlive = nullptr, *active = nullptr, *left = nullptr;
  float2 *x32 = nullptr, *y32 = nullptr;
  void* x16 = nullptr;
  // pinned host memory: the live-system count of the last step, and the
  // systems' norms or residuals
  int* h_live = nullptr;
  double2* h_val = nullptr;
  std::map<int, hipGraphExec_t> graphs;
  std::set<int> ran;  // steps that have run since the graphs were dropped

  void drop_graphs() {
    for (auto& kv : graphs) (void)hipGraphExecDestroy(kv.second);
    graphs.clear();
    ran.clear();
  }
  void release() {
    drop_graphs();
    void* p[] = {V, w, t, partial, h1, h2, hn, H, cs, sn, g, yv, y64, b, x, d, r, pv, tmp,
                 atol, scale, live, kr, nlive, x32, y32, x16};
    for (void* q : p)
      if (q) (void)hipFree(q);
    if (h_live) (void)hipHostFree(h_live);
    if (h_val) (void)hipHostFree(h_val);
    *this = SolveWs();
  }
};
struct Ws {
  SolveWs one, batch;
  ~Ws() {
    one.release();
    batch.release();
  }
};

Ws* ws_of(smh_op* op) {
  if (!op->solver_ws) op->solver_ws = new Ws();
  return static_cast<Ws*>(op->solver_ws);
}

// SMH_GRAPHS=0 in the environment runs the Arnoldi steps as plain launches
bool graphs_enabled() {
  const char* e = getenv("SMH_GRAPHS");
  return !(e && e[0] == '0');
}

// KB right-hand sides x n_seg segments in lockstep, device-side Givens.
template <int KB>
struct Solver {
  smh_op* op;
  smh_ctx* ctx;
  hipStream_t s;
  SolveWs* ws;
  int64_t n, n8, per_part;  // padded length, times KB, elements per particle
  int restart, cap, nsys, nblk;  // cap: restart length that the workspace's arrays are laid out for
  bool use_P, small;
  int64_t mv64 = 0, mv32 = 0, mv16 = 0, iters = 0;

  int init() {
    nsys = op->n_seg * KB;
    // dot partials: about 1024 entries of the largest segment per block, the chip filled at most twice
    int64_t most = 0;
    for (int q = 0; q < op->n_seg; ++q) most = std::max(most, (op->seg_off[q + 1] - op->seg_off[q]) * per_part);
    nblk = (int)std::max<int64_t>(1, std::min<int64_t>((most + 1023) / 1024, std::max(8, kDotBlocks / op->n_seg)));
    use_P = op->d_P != nullptr;
    small = KB == 1 && op->n_seg == 1 && n8 <= kSmallVector;
    cap = std::max(restart, ws->restart);
    if (ws->n8 == n8 && ws->restart >= restart && ws->nsys == nsys && ws->nblk == nblk) return SMH_OK;
    cap = restart;
    ws->release();
    const size_t n32 = KB == 1 ? (size_t)n : (size_t)op->n_part * op->b32_S * KB;
    const bool half = KB > 1 && smh::op_has_batch(op, SMH_FP16);
    const int ldh = restart + 1;
    auto alloc = [&](void** p, size_t bytes) { return hipMalloc(p, std::max<size_t>(bytes, 16)) == hipSuccess; };
    const bool ok =
        alloc((void**)&ws->V, (size_t)(restart + 1) * n8 * sizeof(double2)) &&
        alloc((void**)&ws->w, n8 * sizeof(double2)) && alloc((void**)&ws->t, n * sizeof(double2)) &&
        alloc((void**)&ws->partial, (size_t)op->n_seg * nblk * kMaxBasis * KB * sizeof(double2)) &&
        alloc((void**)&ws->h1, (size_t)nsys * ldh * sizeof(double2)) &&
        alloc((void**)&ws->h2, (size_t)nsys * ldh * sizeof(double2)) &&
        alloc((void**)&ws->hn, (size_t)nsys * sizeof(double2)) &&
        alloc((void**)&ws->H, (size_t)nsys * (restart + 1) * restart * sizeof(double2)) &&
        alloc((void**)&ws->cs, (size_t)nsys * restart * sizeof(double2)) &&
        alloc((void**)&ws->sn, (size_t)nsys * restart * sizeof(double2)) &&
        alloc((void**)&ws->g, (size_t)nsys * (restart + 1) * sizeof(double2)) &&
        alloc((void**)&ws->yv, (size_t)nsys * ldh * sizeof(double2)) &&
        alloc((void**)&ws->y64, n8 * sizeof(double2)) && alloc((void**)&ws->b, n8 * sizeof(double2)) &&
        alloc((void**)&ws->x, n8 * sizeof(double2)) && alloc((void**)&ws->d, n8 * sizeof(double2)) &&
        alloc((void**)&ws->r, n8 * sizeof(double2)) &&
        (KB == 1 || (alloc((void**)&ws->pv, n8 * sizeof(double2)) && alloc((void**)&ws->tmp, n8 * sizeof(double2)))) &&
        alloc((void**)&ws->atol, 3 * nsys * sizeof(double)) && alloc((void**)&ws->scale, nsys * sizeof(double)) &&
        alloc((void**)&ws->live, nsys * sizeof(int)) && alloc((void**)&ws->kr, nsys * sizeof(int)) &&
        alloc((void**)&ws->nlive, (restart + 1) * sizeof(int)) &&
        alloc((void**)&ws->x32, n32 * sizeof(float2)) && alloc((void**)&ws->y32, n8 * sizeof(float2)) &&
        (!half || alloc(&ws->x16, n32 * 2 * sizeof(_Float16))) &&
        hipHostMalloc((void**)&ws->h_live, 4 * sizeof(int), hipHostMallocDefault) == hipSuccess &&
        hipHostMalloc((void**)&ws->h_val, (size_t)nsys * sizeof(double2), hipHostMallocDefault) == hipSuccess;
    if (!ok) {
      ws->release();
      return smh_fail(ctx, SMH_ERR_HIP, "solver allocation failed (%lld entries, restart %d)", (long long)n8, restart);
    }
    ws->res = ws->atol + nsys;
    ws->left = (int*)(ws->res + nsys);
    ws->active = ws->left + nsys;
    // the FP32 input's padding slots stay zero
    hipLaunchKernelGGL(zero_f2_kernel, dim3(1024), dim3(256), 0, s, ws->x32, (int64_t)n32);
    SMH_HIP(ctx, hipGetLastError());
    ws->n8 = n8;
    ws->restart = restart;
    ws->nsys = nsys;
    ws->nblk = nblk;
    return SMH_OK;
  }

  int apply(int precision, const void* x, void* y) {
    return KB == 1 ? smh::op_apply(op, precision, x, y, false) : smh::op_apply_batch(op, precision, x, y, false);
  }

  // out = M v, or M P v with the preconditioner (with_P)
  int master(const double2* v, double2* out, int precision, bool with_P) {
    int rc;
    const double2* src = v;
    if (with_P) {
      if ((rc = smh::op_apply_precond_batch(op, v, ws->pv, false))) return rc;
      src = ws->pv;
    }
    if (precision == SMH_FP64) {
      if ((rc = apply(SMH_FP64, src, ws->y64))) return rc;
      hipLaunchKernelGGL(bmaster_fp64_kernel<KB>, dim3(blocks_for(n8)), dim3(256), 0, s, src, ws->t, ws->y64, out, n8);
      ++mv64;
    } else if (precision == SMH_FP16) {
      if ((rc = smh::op_to_half_batch(op, src, ws->x16))) return rc;
      if ((rc = apply(SMH_FP16, ws->x16, ws->y32))) return rc;
      hipLaunchKernelGGL(bmaster_fp32_kernel<KB>, dim3(blocks_for(n8)), dim3(256), 0, s, src, ws->t, ws->y32, out, n8);
      ++mv16;
    } else {
      if (KB == 1)
        hipLaunchKernelGGL(to_fp32_kernel, dim3(blocks_for(n8)), dim3(256), 0, s, src, ws->x32, n8);
      else
        hipLaunchKernelGGL(to_fp32_b32_kernel, dim3(blocks_for(n8)), dim3(256), 0, s, src, ws->x32, n8, op->B,
                           op->b32_S, (const int*)op->d_b32_tab);
      if ((rc = apply(SMH_FP32, ws->x32, ws->y32))) return rc;
      hipLaunchKernelGGL(bmaster_fp32_kernel<KB>, dim3(blocks_for(n8)), dim3(256), 0, s, src, ws->t, ws->y32, out, n8);
      ++mv32;
    }
    SMH_HIP(ctx, hipGetLastError());
    return SMH_OK;
  }

  // out[sys * ldo + j] = V_j[., sys]^H w[., sys], j < nv (device, no sync)
  int dots(const double2* Vb, int nv, const double2* wv, double2* out, int ldo) {
    if (nv < 1 || nv > kMaxBasis) return smh_fail(ctx, SMH_ERR_ARG, "basis size out of range");
    hipLaunchKernelGGL(sdot_kernel<KB>, dim3(nblk, op->n_seg), dim3(kDotThreads), 0, s, Vb, n8, nv, wv, per_part,
                       (const int64_t*)op->d_seg_off, ws->partial);
    hipLaunchKernelGGL(sreduce_kernel<KB>, dim3(nv * KB, op->n_seg), dim3(256), 0, s, ws->partial, nblk, out, ldo);
    SMH_HIP(ctx, hipGetLastError());
    return SMH_OK;
  }
  // ||v|| of every system, to the host
  int norms(const double2* v, double* out) {
    int rc = dots(v, 1, v, ws->hn, 1);
    if (rc) return rc;
    SMH_HIP(ctx, hipMemcpyAsync(ws->h_val, ws->hn, nsys * sizeof(double2), hipMemcpyDeviceToHost, s));
    SMH_HIP(ctx, hipStreamSynchronize(s));
    for (int k = 0; k < nsys; ++k) out[k] = std::sqrt(std::max(0.0, ws->h_val[k].x));
    return SMH_OK;
  }

  void saxpy(int nv, const double2* c, double sgn, double2* w) {
    hipLaunchKernelGGL(saxpy_kernel<KB>, dim3(blocks_for(n8)), dim3(256), 0, s, ws->V, n8, nv, c, cap + 1, sgn, w,
                       n8, per_part, (const int*)op->d_seg_of);
  }

  // Arnoldi step k of every system: w = M (P) V_k, CGS2, ||w||, rotation,
  // V_{k+1} = w / ||w||, the live count to the host. Device only (captured in
  // a graph).
  int arnoldi_step(int k, int precision) {
    int rc;
    const int ldh = cap + 1;
    const double2* vk = ws->V + (size_t)k * n8;
    if ((rc = master(vk, ws->w, precision, use_P))) return rc;
    if (small && (k + 1) * n8 <= kSmallBasis) {
      hipLaunchKernelGGL(arnoldi_small_kernel, dim3(1), dim3(kSmallThreads), 0, s, k, ws->V, (const double2*)ws->w,
                         (int)n8, ws->atol, ws->left, cap, ws->live, ws->H, ws->cs, ws->sn, ws->g, ws->kr, ws->nlive,
                         ws->h_live);
      SMH_HIP(ctx, hipGetLastError());
      return SMH_OK;
    }
    if ((rc = dots(ws->V, k + 1, ws->w, ws->h1, ldh))) return rc;
    saxpy(k + 1, ws->h1, -1.0, ws->w);
    if ((rc = dots(ws->V, k + 1, ws->w, ws->h2, ldh))) return rc;
    saxpy(k + 1, ws->h2, -1.0, ws->w);
    if ((rc = dots(ws->w, 1, ws->w, ws->hn, 1))) return rc;
    hipLaunchKernelGGL(givens_kernel, dim3(blocks_for(nsys, 64)), dim3(64), 0, s, k, ws->h1, ws->h2, ldh, ws->hn,
                       ws->atol, ws->left, nsys, cap, ws->live, ws->H, ws->cs, ws->sn, ws->g, ws->kr, ws->scale, ws->nlive);
    hipLaunchKernelGGL(sscale_kernel<KB>, dim3(blocks_for(n8)), dim3(256), 0, s, ws->w, ws->scale,
                       ws->V + (size_t)(k + 1) * n8, n8, per_part, (const int*)op->d_seg_of,
                       (const int*)(ws->nlive + k), ws->h_live);
    SMH_HIP(ctx, hipGetLastError());
    return SMH_OK;
  }

  // Step k: its first run is eager (lazy allocations and kernel attributes
  // happen outside any capture, and a solver used once pays for no graph), the
  // second is captured and replayed from then on.
  int run_step(int k, int precision) {
    const int pi = precision == SMH_FP64 ? 0 : (precision == SMH_FP32 ? 1 : 2);
    const int ui = use_P ? 1 : 0;
    const int key = ((pi * 2 + ui) << 8) | k;
    if (!graphs_enabled() || !ws->ran.count(key)) {
      const int rc = arnoldi_step(k, precision);
      if (!rc) ws->ran.insert(key);
      return rc;
    }
    auto it = ws->graphs.find(key);
    if (it == ws->graphs.end()) {
      // the matvec counters count launches: the replay below counts this step's one matvec
      const int64_t c64 = mv64, c32 = mv32, c16 = mv16;
      // recorded on the stream that only captures use: threads with other operators share the context's other one,
      // whose work would end up in this graph, and whose synchronizations fail, during the capture
      std::unique_lock<std::mutex> one(*ctx->capture_lock);
      SMH_HIP(ctx, hipStreamBeginCapture(ctx->capture, hipStreamCaptureModeRelaxed));
      smh_ctx* const home = ctx;
      smh_ctx recording = *ctx;
      recording.stream = s = ctx->capture;
      op->ctx = ctx = &recording;
      const int rc = arnoldi_step(k, precision);
      op->ctx = ctx = home;
      s = ctx->stream;
      if (rc) ctx->last_error = recording.last_error;
      mv64 = c64;
      mv32 = c32;
      mv16 = c16;
      hipGraph_t graph = nullptr;
      const hipError_t e = hipStreamEndCapture(ctx->capture, &graph);
      one.unlock();
      if (rc || e != hipSuccess) {
        if (graph) (void)hipGraphDestroy(graph);
        return rc ? rc : smh_fail(ctx, SMH_ERR_HIP, "graph capture failed: %s", hipGetErrorString(e));
      }
      hipGraphExec_t exec = nullptr;
      const hipError_t ei = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
      (void)hipGraphDestroy(graph);
      if (ei != hipSuccess) return smh_fail(ctx, SMH_ERR_HIP, "graph instantiation failed: %s", hipGetErrorString(ei));
      it = ws->graphs.emplace(key, exec).first;
    }
    SMH_HIP(ctx, hipGraphLaunch(it->second, s));
    if (precision == SMH_FP64)
      ++mv64;
    else if (precision == SMH_FP16)
      ++mv16;
    else
      ++mv32;
    return SMH_OK;
  }

  // the systems' residuals (or estimates) and steps left to the host
  int residuals(double* res_out, int* left) {
    SMH_HIP(ctx, hipMemcpyAsync(ws->h_val, ws->res, nsys * (sizeof(double) + sizeof(int)), hipMemcpyDeviceToHost, s));
    SMH_HIP(ctx, hipStreamSynchronize(s));
    const double* v = reinterpret_cast<const double*>(ws->h_val);
    std::copy(v, v + nsys, res_out);
    std::copy((const int*)(v + nsys), (const int*)(v + nsys) + nsys, left);
    return SMH_OK;
  }

  // GMRES on M x = b for the systems with active[sys] (others left untouched)
  // from x (in/out), each to ||b - M x|| <= atol[sys]. x_zero: x is zero on
  // entry, so the first residual is b itself. trust_estimate (inner solves of
  // the refinement): one restart cycle at most, returning as soon as the
  // Arnoldi residual estimates reach atol or the cycle ends, without
  // recomputing the true residual (the caller takes it in FP64 and starts the
  // next sweep: a reduced-precision operator whose error sits above atol would
  // otherwise stall the restarts). left[sys]: steps the system may take, and
  // may still take afterwards: on lookup operators the systems share the count
  // of the steps taken together, on the explicit matrix each counts its own
  // (there right-hand sides solved one after the other had maxiter each, and
  // one that ends a sweep early must not pay for the others' steps).
  // res_out[sys]: residual of x (or the estimate); steps: Arnoldi steps taken.
  int gmres(double2* x, const double2* b, const double* atol, const int* active, int* left, int precision,
            double* res_out, int& steps, bool x_zero, bool trust_estimate) {
    int rc;
    std::vector<double> systems(3 * (size_t)nsys, 0.0);
    std::copy(atol, atol + nsys, systems.data());
    std::copy(left, left + nsys, (int*)(systems.data() + 2 * nsys));
    std::copy(active, active + nsys, (int*)(systems.data() + 2 * nsys) + nsys);
    SMH_HIP(ctx, hipMemcpyAsync(ws->atol, systems.data(), systems.size() * sizeof(double), hipMemcpyHostToDevice, s));
    steps = 0;
    for (int outer = 0;; ++outer) {
      if (outer == 0 && x_zero) {
        SMH_HIP(ctx, hipMemcpyAsync(ws->w, b, n8 * sizeof(double2), hipMemcpyDeviceToDevice, s));
      } else {
        if ((rc = master(x, ws->w, precision, false))) return rc;
        hipLaunchKernelGGL(sub_kernel, dim3(blocks_for(n8)), dim3(256), 0, s, b, ws->w, ws->w, n8);
      }
      if ((rc = dots(ws->w, 1, ws->w, ws->hn, 1))) return rc;
      hipLaunchKernelGGL(zero_int_kernel, dim3(1), dim3(256), 0, s, ws->nlive, cap + 1);
      hipLaunchKernelGGL(cycle_init_kernel, dim3(blocks_for(nsys, 64)), dim3(64), 0, s, ws->hn, ws->atol, ws->active,
                         ws->left, nsys, cap, ws->g, ws->live, ws->scale, ws->res, ws->kr, ws->nlive);
      // V_0 (zero for systems that do not run) and the live count
      hipLaunchKernelGGL(sscale_kernel<KB>, dim3(blocks_for(n8)), dim3(256), 0, s, ws->w, ws->scale, ws->V, n8,
                         per_part, (const int*)op->d_seg_of, (const int*)(ws->nlive + cap), ws->h_live);
      SMH_HIP(ctx, hipGetLastError());
      if ((rc = residuals(res_out, left))) return rc;
      if (ws->h_live[0] == 0) return SMH_OK;
      int k = 0;
      for (; k < restart; ++k, ++steps) {
        if ((rc = run_step(k, precision))) return rc;
        ++iters;
        SMH_HIP(ctx, hipStreamSynchronize(s));
        if (*(volatile int*)ws->h_live == 0) {
          ++k;
          ++steps;
          break;
        }
      }
      // y = R^-1 g per system, then x += V y (or x += P V y) for all at once
      hipLaunchKernelGGL(backsub_kernel, dim3(blocks_for(nsys, 64)), dim3(64), 0, s, nsys, cap, ws->H, ws->g, ws->kr,
                         ws->yv, cap + 1, ws->res, op->kind == 2 ? -1 : k, ws->left);
      if (k > 0) {
        if (use_P) {
          hipLaunchKernelGGL(zero2_kernel, dim3(1024), dim3(256), 0, s, ws->tmp, n8);
          saxpy(k, ws->yv, 1.0, ws->tmp);
          if ((rc = smh::op_apply_precond_batch(op, ws->tmp, x, true))) return rc;
        } else {
          saxpy(k, ws->yv, 1.0, x);
        }
      }
      SMH_HIP(ctx, hipGetLastError());
      if (trust_estimate) return residuals(res_out, left);
    }
  }
};

}  // namespace

namespace smh {

void solver_release(smh_op* op) {
  if (op->solver_ws) delete static_cast<Ws*>(op->solver_ws);
  op->solver_ws = nullptr;
}

void solver_drop_graphs(smh_op* op) {
  if (!op->solver_ws) return;
  static_cast<Ws*>(op->solver_ws)->one.drop_graphs();
  static_cast<Ws*>(op->solver_ws)->batch.drop_graphs();
}

int op_apply_precond_batch(smh_op* op, const double2* x, double2* y, bool accumulate) {
  smh_ctx* ctx = op->ctx;
  SMH_CHECK(ctx, op->d_P != nullptr && op->d_Pnbr != nullptr, SMH_ERR_STATE, "no preconditioner set");
  SMH_CHECK(ctx, op->B * kB <= 512, SMH_ERR_UNSUPPORTED, "blocksize too large for the preconditioner kernel");
  const size_t lds = (size_t)op->B * kB * sizeof(double2);
  hipLaunchKernelGGL(precond_kernel, dim3((unsigned)op->n_part), dim3(256), lds, ctx->stream, (const double2*)op->d_P,
                     (const int*)op->d_Pnbr, op->P_k1, x, y, op->B, accumulate ? 1 : 0);
  SMH_HIP(ctx, hipGetLastError());
  return SMH_OK;
}

int op_reserve_precond(smh_op* op, int k1) {
  smh_ctx* ctx = op->ctx;
  if (op->d_P && op->P_k1 == k1) return SMH_OK;
  SMH_HIP(ctx, hipStreamSynchronize(ctx->stream));
  solver_drop_graphs(op);  // graphs hold the buffers' addresses
  if (op->d_P) (void)hipFree(op->d_P);
  if (op->d_Pnbr) (void)hipFree(op->d_Pnbr);
  op->d_P = nullptr;
  op->d_Pnbr = nullptr;
  op->P_k1 = 0;
  SMH_HIP(ctx, hipMalloc(&op->d_P, (size_t)op->n_part * k1 * op->B * op->B * sizeof(double2)));
  SMH_HIP(ctx, hipMalloc(&op->d_Pnbr, (size_t)op->n_part * k1 * sizeof(int)));
  op->P_k1 = k1;
  return SMH_OK;
}

}  // namespace smh

// Blocks of KB right-hand sides over every segment, solved together (every
// coupling matvec is one launch for all systems).
template <int KB>
static int solve_blocks(smh_op* op, const double* t_diag, const double* rhs, double* x, int64_t nrhs, double tol,
                        int restart, int maxiter, int mode, double* stats,
                        std::chrono::steady_clock::time_point t0) {
  smh_ctx* ctx = op->ctx;
  hipStream_t s = ctx->stream;
  Ws* all = ws_of(op);
  Solver<KB> S;
  S.op = op;
  S.ctx = ctx;
  S.s = s;
  S.ws = KB == 1 ? &all->one : &all->batch;
  S.n = op->n_part * op->B;
  S.n8 = S.n * KB;
  S.per_part = (int64_t)op->B * KB;
  S.restart = restart;
  int rc = S.init();
  if (rc) return rc;
  SolveWs* ws = S.ws;
  const int nsys = S.nsys;
  if ((rc = smh::op_reserve_packed(op, KB))) return rc;
  if (KB > 1 && (rc = smh::op_reserve_batch(op))) return rc;
  SMH_HIP(ctx, hipMemcpyAsync(op->d_pk_in, t_diag, op->n_unk * sizeof(double2), hipMemcpyDefault, s));
  if ((rc = smh::op_unpack(op, SMH_FP64, op->d_pk_in, ws->t))) return rc;
  double worst = 0, sweeps_total = 0;
  int64_t steps_total = 0;
  bool converged_all = true;
  std::vector<double> bnorm(nsys), atol(nsys), res(nsys), prev_res(nsys), inner_atol(nsys), inner_res(nsys);
  std::vector<int> active(nsys), act(nsys), left(nsys);
  for (int64_t r0 = 0; r0 < nrhs; r0 += KB) {
    const int nb = (int)std::min<int64_t>(KB, nrhs - r0);
    SMH_HIP(ctx, hipMemcpyAsync(op->d_pk_in, rhs + 2 * r0 * op->n_unk, (size_t)nb * op->n_unk * sizeof(double2),
                                hipMemcpyDefault, s));
    if ((rc = KB == 1 ? smh::op_unpack(op, SMH_FP64, op->d_pk_in, ws->b)
                      : smh::op_unpack_batch(op, SMH_FP64, op->d_pk_in, nb, ws->b)))
      return rc;
    if ((rc = S.norms(ws->b, bnorm.data()))) return rc;
    for (int q = 0; q < nsys; ++q) {
      atol[q] = tol * bnorm[q];
      active[q] = (q % KB) < nb && bnorm[q] > 0.0;
    }
    std::fill(left.begin(), left.end(), maxiter);
    int steps = 0;
    if (mode == SMH_SOLVE_FP64) {
      // x0 = rhs, as smuthi passes rhs as initial guess
      SMH_HIP(ctx, hipMemcpyAsync(ws->x, ws->b, S.n8 * sizeof(double2), hipMemcpyDeviceToDevice, s));
      if ((rc = S.gmres(ws->x, ws->b, atol.data(), active.data(), left.data(), SMH_FP64, res.data(), steps, false, false)))
        return rc;
      steps_total += steps;
      sweeps_total += 1;
    } else {
      hipLaunchKernelGGL(zero2_kernel, dim3(1024), dim3(256), 0, s, ws->x, S.n8);
      SMH_HIP(ctx, hipMemcpyAsync(ws->r, ws->b, S.n8 * sizeof(double2), hipMemcpyDeviceToDevice, s));
      for (int q = 0; q < nsys; ++q) res[q] = bnorm[q];
      bool fresh = true;
      bool fp64_residuals = mode != SMH_SOLVE_MIXED16;
      const int inner_prec = mode == SMH_SOLVE_MIXED16 ? SMH_FP16 : SMH_FP32;
      for (int sweep = 0; sweep < 50; ++sweep) {
        if (sweep > 0) {
          // FP16 inner solves: the residual that drives the next sweep comes
          // from the FP32 matvec (accurate to a few 1e-7 of ||b||, far below
          // the FP16 sweep's own error) while it is well above that floor;
          // once it meets the tolerance or nears the floor, FP64 residuals
          // certify the result and drive any further sweeps
          bool certified = fp64_residuals;
          if (!certified) {
            if ((rc = S.master(ws->x, ws->r, SMH_FP32, false))) return rc;
            hipLaunchKernelGGL(sub_kernel, dim3(blocks_for(S.n8)), dim3(256), 0, s, ws->b, ws->r, ws->r, S.n8);
            if ((rc = S.norms(ws->r, res.data()))) return rc;
            bool need64 = false, last = true;
            for (int q = 0; q < nsys; ++q) {
              if (!active[q]) continue;
              need64 = need64 || res[q] <= std::max(atol[q], kFp32ResidualFloor * bnorm[q]);
              // the next sweep gains about the factor this one did: if that
              // takes every system to the tolerance or to the FP32 floor, its
              // residual is taken in FP64 directly
              last = last && prev_res[q] > 0.0 &&
                     res[q] * (res[q] / prev_res[q]) <= std::max(0.5 * atol[q], kFp32ResidualFloor * bnorm[q]);
            }
            certified = need64;
            fp64_residuals = need64 || last;
          }
          if (certified) {
            if ((rc = S.master(ws->x, ws->r, SMH_FP64, false))) return rc;
            hipLaunchKernelGGL(sub_kernel, dim3(blocks_for(S.n8)), dim3(256), 0, s, ws->b, ws->r, ws->r, S.n8);
            if ((rc = S.norms(ws->r, res.data()))) return rc;
            fresh = true;
          }
        }
        bool any = false;
        for (int q = 0; q < nsys; ++q) {
          prev_res[q] = res[q];
          act[q] = active[q] && res[q] > atol[q] && left[q] > 0;
          inner_atol[q] = std::max(atol[q] * 0.5, (mode == SMH_SOLVE_MIXED16 ? kInnerRel16 : kInnerRel) * res[q]);
          any = any || act[q];
        }
        if (!any) break;
        hipLaunchKernelGGL(zero2_kernel, dim3(1024), dim3(256), 0, s, ws->d, S.n8);
        int inner_steps = 0;
        if ((rc = S.gmres(ws->d, ws->r, inner_atol.data(), act.data(), left.data(), inner_prec, inner_res.data(),
                          inner_steps, true, true)))
          return rc;
        steps_total += inner_steps;
        hipLaunchKernelGGL(add_kernel, dim3(blocks_for(S.n8)), dim3(256), 0, s, ws->x, ws->d, S.n8);
        sweeps_total += 1;
        fresh = false;
      }
      if (!fresh) {
        if ((rc = S.master(ws->x, ws->r, SMH_FP64, false))) return rc;
        hipLaunchKernelGGL(sub_kernel, dim3(blocks_for(S.n8)), dim3(256), 0, s, ws->b, ws->r, ws->r, S.n8);
        if ((rc = S.norms(ws->r, res.data()))) return rc;
      }
    }
    for (int q = 0; q < nsys; ++q) {
      if ((q % KB) >= nb) continue;
      const double rel = bnorm[q] > 0 ? res[q] / bnorm[q] : 0.0;
      worst = std::max(worst, rel);
      if (rel > tol) converged_all = false;
    }
    if ((rc = KB == 1 ? smh::op_pack(op, SMH_FP64, ws->x, op->d_pk_out)
                      : smh::op_pack_batch(op, SMH_FP64, ws->x, nb, op->d_pk_out)))
      return rc;
    SMH_HIP(ctx, hipMemcpyAsync(x + 2 * r0 * op->n_unk, op->d_pk_out, (size_t)nb * op->n_unk * sizeof(double2),
                                hipMemcpyDefault, s));
  }
  SMH_HIP(ctx, hipStreamSynchronize(s));
  const double secs = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  if (stats) {
    stats[0] = (double)steps_total;
    stats[1] = (double)S.mv64;
    stats[2] = (double)S.mv32;
    stats[3] = worst;
    stats[4] = secs;
    stats[5] = sweeps_total;
    stats[6] = KB == 1 ? 0.0 : (double)KB;  // right-hand sides per batched matvec
    stats[7] = (double)S.mv16;
  }
  if (!converged_all)
    return smh_fail(ctx, SMH_ERR_NOCONV, "GMRES stopped at relative residual %.3e (tol %.1e)", worst, tol);
  return SMH_OK;
}

extern "C" int smh_solve(smh_op* op, const double* t_diag, const double* rhs, double* x, int64_t nrhs, double tol,
                         int restart, int maxiter, int mode, double* stats) {
  if (!op) return SMH_ERR_ARG;
  smh_ctx* ctx = op->ctx;
  SMH_CHECK(ctx, t_diag && rhs && x && nrhs >= 1, SMH_ERR_ARG, "invalid solve arguments");
  SMH_CHECK(ctx, mode == SMH_SOLVE_FP64 || mode == SMH_SOLVE_MIXED || mode == SMH_SOLVE_MIXED16 || mode == SMH_SOLVE_LU,
            SMH_ERR_ARG, "invalid mode %d", mode);
  if (mode == SMH_SOLVE_LU) {
    SMH_HIP(ctx, hipSetDevice(ctx->device));
    return smh::lu_solve(op, t_diag, rhs, x, nrhs, stats);
  }
  SMH_CHECK(ctx, tol > 0 && restart >= 1 && restart < kMaxBasis && maxiter >= 1, SMH_ERR_ARG,
            "invalid tolerance / restart / maxiter");
  SMH_CHECK(ctx, mode != SMH_SOLVE_MIXED16 || (smh::op_has_batch(op, SMH_FP16) && smh::op_has_batch(op, SMH_FP64)),
            SMH_ERR_UNSUPPORTED, "FP16-operand solves need a lookup operator with the batched FP16 kernel");
  SMH_CHECK(ctx, op->has_table, SMH_ERR_STATE, "coupling table not set");
  SMH_HIP(ctx, hipSetDevice(ctx->device));
  const auto t0 = std::chrono::steady_clock::now();
  const bool batch_ok = smh::op_has_batch(op, SMH_FP32) && smh::op_has_batch(op, SMH_FP64);
  const bool blocks_ok = smh::op_takes_blocks(op, SMH_FP32) && smh::op_takes_blocks(op, SMH_FP64);
  const bool need_batch = mode == SMH_SOLVE_MIXED16 || op->d_P != nullptr || op->n_seg > 1;
  SMH_CHECK(ctx, batch_ok || !need_batch, SMH_ERR_UNSUPPORTED,
            "ensembles and preconditioned solves need an operator with the batched kernels");
  if (blocks_ok && (nrhs > 1 || need_batch))
    return solve_blocks<kB>(op, t_diag, rhs, x, nrhs, tol, restart, maxiter, mode, stats, t0);
  return solve_blocks<1>(op, t_diag, rhs, x, nrhs, tol, restart, maxiter, mode, stats, t0);
}

extern "C" int smh_op_set_preconditioner(smh_op* op, int k1, const int* nbr, const double* blocks) {
  if (!op) return SMH_ERR_ARG;
  smh_ctx* ctx = op->ctx;
  SMH_HIP(ctx, hipSetDevice(ctx->device));
  if (!blocks) {
    if (op->d_P) {
      SMH_HIP(ctx, hipStreamSynchronize(ctx->stream));
      smh::solver_drop_graphs(op);  // graphs hold the buffers' addresses
      (void)hipFree(op->d_P);
      if (op->d_Pnbr) (void)hipFree(op->d_Pnbr);
      op->d_P = nullptr;
      op->d_Pnbr = nullptr;
      op->P_k1 = 0;
    }
    return SMH_OK;
  }
  SMH_CHECK(ctx, k1 >= 1 && k1 <= 64 && nbr, SMH_ERR_ARG, "invalid preconditioner pattern");
  SMH_CHECK(ctx, smh::op_has_batch(op, SMH_FP32) && smh::op_has_batch(op, SMH_FP64), SMH_ERR_UNSUPPORTED,
            "preconditioned solves need an operator with the batched kernels");
  for (int64_t i = 0; i < op->n_part * k1; ++i)
    SMH_CHECK(ctx, nbr[i] >= -1 && nbr[i] < op->n_part, SMH_ERR_ARG, "emitter index %d out of range", nbr[i]);
  if (int rc = smh::op_reserve_precond(op, k1)) return rc;
  const size_t bytes = (size_t)op->n_part * k1 * op->B * op->B * sizeof(double2);
  SMH_HIP(ctx, hipMemcpyAsync(op->d_P, blocks, bytes, hipMemcpyHostToDevice, ctx->stream));
  SMH_HIP(ctx, hipMemcpyAsync(op->d_Pnbr, nbr, (size_t)op->n_part * k1 * sizeof(int), hipMemcpyHostToDevice,
                              ctx->stream));
  SMH_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return SMH_OK;
}
