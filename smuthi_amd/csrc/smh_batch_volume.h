// Cubic volume-lookup matvecs for kBatchRhs right-hand sides: FP32, FP64 and
// FP16 operands, with the slot order, phases, input and tap-row layouts of
// batch_slots_kernel, batch_slots64_kernel and batch_half_kernel (one fragment
// row per tap row of the volume lookup).
//
// A pair's block is the weighted sum of 16 tap rows (vol_tap_offset,
// vol_tap_weight: 4 z slices of 4 taps), 8 KB each in FP32 at l_max 3: the product is bound by fetching rows,
// not by arithmetic. Sorted by (receiver chunk, bin), as the radial kernels
// need it for their receiver sums in LDS, a bin of a chunk holds 1.3 pairs and
// every pair fetches its own 16 rows, at the 11 TB/s of the caches behind the
// L2. So the pairs are sorted by bin alone (7 pairs per bin for 700 spheres,
// and neighbouring bins share half of their rows or more), each pair's product
// is written out, and vol_sum_kernel adds the products of each receiver: 2 KB
// written and read per pair instead of 128 KB fetched from behind the L2. The
// pairs run in slabs of neighbouring bins, small enough that a slab's products
// are read back from the last-level cache.
//   * All slices in one pass; the taps are summed before the product, one MFMA
//     per K-step (FP16: one per tap, so that the taps are summed in FP32).
//   * A wave's unit is two pairs of a bin (FP64: one), which share the loaded
//     rows; the units of a bin go to different waves, which read its rows from
//     the L2 at the same time (VolWalk).
//   * Rows are loaded in pieces through a ring of NB register buffers that
//     runs on into the next unit's rows, and the next unit, its pairs and
//     inputs are fetched while the current one is worked on.
//   * Tap weights are evaluated one per lane and read as scalars.
// 701 spheres, l_max 3, cubic splines, FP32 (982 k pairs over both tables): 8.9
// ms with a launch per slice on receiver chunks, 4.0 + 0.5 ms (sums) here, the
// rows fetched into the L2 once (0.48 GB per slab) and read from it at 11 TB/s;
// what remains is latency, at two waves per SIMD (256 registers). 6 ensembles,
// 108 k pairs, FP16 operands: 1.5 -> 0.54 ms.
//
// Products of a slab: [pair][MH tiles][64 lanes][4] FP32, lane (q, rr) of tile
// i holding column rr = (rhs, re|im) of slots 16 i + 4 q .. + 3; FP64
// [pair][MH tiles][4][64 lanes], register r holding slot 16 i + 4 r + q.
#pragma once

#include <utility>

#include "smh_batch_half.h"
#include "smh_batch_slots.h"
#include "smh_batch_slots64.h"

namespace smh {

// One launch: a slab, whose first pair is pair0.
struct VolKArgs {
  const void* recs;     // PairRec2<Real> sorted by bin
  const int4* units;    // (first tap row, first pair, pairs, -)
  const int* bounds;    // kVolXcds + 1 bounds of the XCDs' units
  const void* tt;       // tap rows
  const void* x;        // input in slot layout
  void* out;            // products
  const float* xmax;    // FP16: scale of the input
  const float* hscale;  // FP16: scale of each tap row
  int pair0, len_z, vmode;
};

// z slices of a volume lookup (vol_tap_offset), and of the cubic ones here
__host__ __device__ constexpr int vol_slices(int vmode) { return vmode >= 2 ? 4 : 1; }
constexpr int kSlices = 4;

// Largest ring of at most `most` buffers that NU pieces fill evenly: a piece's
// buffer is then known at compile time, also across the end of a pair.
__host__ __device__ constexpr int ring_size(int NU, int most) {
  for (int b = most; b > 1; --b)
    if (NU % b == 0) return b;
  return 1;
}

// f(integral_constant 0), ..., f(integral_constant N - 1): register buffers
// indexed by a unit's piece stay in registers.
template <typename F, int... I>
__device__ __forceinline__ void for_pieces(std::integer_sequence<int, I...>, F&& f) {
  (f(std::integral_constant<int, I>{}), ...);
}

// A unit of work of a wave: up to two pairs of one bin, in scalar registers
// (pairs <= 0: no work).
struct VolUnit {
  int row, first, pairs;
};

// A wave's walk over the units of a slab. XCD x (block mod 8) has the units
// bounds[x] .. bounds[x + 1], and its waves take them in turn: at any time they
// work on neighbouring units, the units of a bin fetch its rows together, and
// each row comes into that XCD's L2 once (480 MB per slab of 61 k pairs, 700
// spheres; with an entry of up to 16 pairs per wave 2400 MB, since the waves'
// rows together are several times the L2). Units cost the same, so waves keep
// in step without a counter (tickets from one counter per XCD: 120 ns each).
// Two stages, so that the load is not waited for where it is issued.
constexpr int kVolXcds = 8;
struct VolWalk {
  const int4* units;
  int next, end, stride;
  int4 en = make_int4(0, 0, 0, 0);
  bool found = false;

  __device__ __forceinline__ VolWalk(const int4* u, const int* bounds) : units(u) {
    const int x = blockIdx.x & (kVolXcds - 1), waves = blockDim.x >> 6;
    stride = (((int)gridDim.x + kVolXcds - 1 - x) / kVolXcds) * waves;
    next = bounds[x] + (int)(blockIdx.x / kVolXcds) * waves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    end = bounds[x + 1];
  }
  __device__ __forceinline__ void fetch() {
    found = next < end;
    if (found) en = units[next];
    next += stride;
  }
  // (without a further unit: row and pair of the last one, addresses stay in bounds)
  __device__ __forceinline__ VolUnit unit() const {
    VolUnit n;
    n.row = __builtin_amdgcn_readfirstlane(en.x);
    n.first = __builtin_amdgcn_readfirstlane(en.y);
    n.pairs = found ? __builtin_amdgcn_readfirstlane(en.z) : 0;
    return n;
  }
};
// Piece before which stage k of the next unit comes (1: its record, 2: its
// pairs, 3: its input): its row is needed from piece NU - NB on.
__host__ __device__ constexpr int vol_stage(int NU, int NB, int k) {
  return k == 1 ? 0 : (k == 2 ? (NU / 3 < NU - NB ? NU / 3 : NU - NB) : 2 * NU / 3);
}

// Address of a tap row, in scalar registers (rows are the same for all lanes):
// opaque, so that the lane's offset stays a 32-bit register of its own and no
// per-row addresses are kept in vector registers.
typedef __attribute__((address_space(1))) const char* GlobalBytes;
__device__ __forceinline__ GlobalBytes vol_row(const void* tt, int row, unsigned row_bytes) {
  GlobalBytes r = (GlobalBytes)tt + (size_t)(unsigned)row * row_bytes;
  asm volatile("" : "+s"(r));
  return r;
}
template <typename V>
__device__ __forceinline__ V vol_load(GlobalBytes r, unsigned lane_off, unsigned at) {
  asm volatile("" : "+v"(lane_off));
  return *reinterpret_cast<__attribute__((address_space(1))) const V*>(r + lane_off + at);
}
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef double f64x2_t __attribute__((ext_vector_type(2)));
typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));

__device__ inline float lane_value(float v, int l) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l)); }
__device__ inline double lane_value(double v, int l) {
  const long long b = __double_as_longlong(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(b & 0xffffffffLL), l);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(b >> 32), l);
  return __longlong_as_double(((long long)hi << 32) | lo);
}

// Tap weight of lane 4 s + t for slice s, tap t
template <typename Real>
__device__ inline Real vol_lane_weight(int vmode, int lane, Real w, Real w2) {
  return vol_tap_weight<Real>(vmode, (lane >> 2) & 3, lane & 3, w, w2);
}

constexpr int kVolRing32 = 4, kVolRing64 = 4, kVolRingHalf = 4;
// Pairs of a unit: FP32 and FP16 operands, FP64.
constexpr int kVolPairs32 = 2, kVolPairs64 = 1;

// Workgroup of four waves, two waves per SIMD: 256 registers per lane.
constexpr int kVolThreads = 256;

// Receiver phase of a lane's four rows (slot group 4 i + q of tile i): (cos,
// sin) of |m| phi, by the weights hq[k] = [q == k] (selects between the array's
// elements would put it into scratch memory), and the sign masks of rows 0, 1
// and 2, 3.
template <int LMAX, int MMAX, int i>
__device__ __forceinline__ void row_phase(int q, const float (&hq)[4], const float (&cs)[MMAX + 1],
                                          const float (&sn)[MMAX + 1], float& c, float& s, unsigned& lo, unsigned& hi) {
  constexpr SlotOrder<LMAX, MMAX> so{};
  constexpr int m0 = so.absm[4 * i], m1 = so.absm[4 * i + 1], m2 = so.absm[4 * i + 2], m3 = so.absm[4 * i + 3];
  constexpr int s0 = so.sgn[4 * i], s1 = so.sgn[4 * i + 1], s2 = so.sgn[4 * i + 2], s3 = so.sgn[4 * i + 3];
  constexpr unsigned neg = (s0 < 0) | (s1 < 0) << 1 | (s2 < 0) << 2 | (s3 < 0) << 3;
  constexpr unsigned pos = (s0 > 0) | (s1 > 0) << 1 | (s2 > 0) << 2 | (s3 > 0) << 3;
  c = hq[0] * cs[m0];
  c = fmaf(hq[1], cs[m1], c);
  c = fmaf(hq[2], cs[m2], c);
  c = fmaf(hq[3], cs[m3], c);
  s = hq[0] * sn[m0];
  s = fmaf(hq[1], sn[m1], s);
  s = fmaf(hq[2], sn[m2], s);
  s = fmaf(hq[3], sn[m3], s);
  lo = (neg >> q) << 31;
  hi = (~pos >> q) << 31;
}

// ---- FP32 -------------------------------------------------------------------
// A piece is four K-steps of one tile for the four taps of one slice (16
// registers).
template <int LMAX, int MMAX>
__global__ void __launch_bounds__(kVolThreads, 2) vol_slots_kernel(VolKArgs a) {
  using Sh = SlotShape<LMAX, MMAX, 4>;
  constexpr int S = Sh::S, NS = Sh::NS, MT = Sh::MT, MH = Sh::MH;
  constexpr int KB = kBatchRhs, N4 = NS / 4, G = kVolPairs32;
  constexpr int NU = MT * N4 * kSlices, NB = ring_size(NU, kVolRing32);
  static_assert(KB * 2 == 16, "16 result columns = kBatch right-hand sides x (re, im)");
  static_assert(NS % 4 == 0, "whole float4 groups of K-steps");
  static_assert(MMAX <= 4, "phase selection covers |m| <= 4");
  constexpr SlotOrder<LMAX, MMAX> so{};
  static_assert(so.ok, "slot order");
  using Rec = PairRec2<float>;
  using V4 = typename Mfma<float>::v4;

  const int lane = threadIdx.x & 63;
  const Rec* recs = reinterpret_cast<const Rec*>(a.recs);
  const float2* xg = reinterpret_cast<const float2*>(a.x);

  const int rr = lane & 15, q = lane >> 4;
  const int rhs = rr >> 1, zp = rr & 1;
  const float hq[4] = {q == 0 ? 1.f : 0.f, q == 1 ? 1.f : 0.f, q == 2 ? 1.f : 0.f, q == 3 ? 1.f : 0.f};
  const unsigned zmask = zp ? 0u : 0x80000000u;      // z: sign of the b term for the re column
  const unsigned qmask = q >= 2 ? 0x80000000u : 0u;  // mixed-sign steps: slots 2, 3 have m < 0
  const float sgnz = zp ? 1.f : -1.f;
  const int64_t xlane = (int64_t)(q * KB + rhs) * NS;

  const unsigned lane16 = 16u * (unsigned)lane;
  f32x4_t buf[NB][4];
  // piece u: slice u % kSlices, K-steps 4 s4 .. 4 s4 + 3 of a tile; the Re and the Im tile of a row group in turn
  // (the first piece of each slice sets its rows' addresses)
  GlobalBytes rows[kSlices][4];
  auto load_piece = [&](int row, int u, f32x4_t (&b)[4]) __attribute__((always_inline)) {
    const int sl = u % kSlices, s4 = (u / kSlices) % N4, ti = u / (kSlices * N4);
    const int tile = (ti >> 1) + (ti & 1) * MH;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      if (u < kSlices) rows[sl][t] = vol_row(a.tt, row + vol_tap_offset(a.vmode, sl, t, a.len_z), Sh::FRB * 4);
      b[t] = vol_load<f32x4_t>(rows[sl][t], lane16, (tile * N4 + s4) * 1024);
    }
  };
  auto load_x = [&](const Rec& r, float4 (&xs)[NS / 2]) {
    const float4* xp = reinterpret_cast<const float4*>(xg + (int64_t)(r.ij & kPairMask) * S * KB + xlane);
#pragma unroll
    for (int k = 0; k < NS / 2; ++k) xs[k] = xp[k];
  };

  VolWalk walk(a.units, a.bounds);
  VolUnit cur, nxt;
  Rec rec[G];
  float4 xc[G][NS / 2];
  walk.fetch();
  nxt = walk.unit();
  if (nxt.pairs <= 0) return;
#pragma unroll
  for (int g = 0; g < G; ++g) rec[g] = recs[nxt.first + (g < nxt.pairs ? g : 0)];
#pragma unroll
  for (int u = 0; u < NB; ++u) load_piece(nxt.row, u, buf[u]);
#pragma unroll
  for (int g = 0; g < G; ++g) load_x(rec[g], xc[g]);

  // one unit: two pairs of the current entry (the last one twice where it has an odd number),
  // and the loads of the next unit
  for (;;) {
    cur = nxt;
    if (cur.pairs <= 0) break;
    float cs[G][MMAX + 1], sn[G][MMAX + 1], z[G][NS], wt[G][kSlices * 4];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const float wl = vol_lane_weight<float>(a.vmode, lane, rec[g].w, rec[g].w2);
#pragma unroll
      for (int k = 0; k < kSlices * 4; ++k) wt[g][k] = lane_value(wl, k);
      phase_powers<MMAX>(rec[g].c, rec[g].s, cs[g], sn[g]);
      // B operand per K-step: (e^{i m2 phi} x[slot 4 s + q][rhs]).re or .im
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        const float4 x4 = xc[g][s >> 1];
        const float xr = (s & 1) ? x4.z : x4.x, xi = (s & 1) ? x4.w : x4.y;
        const float av0 = zp ? xi : xr, bv0 = zp ? xr : xi;
        const int am = so.absm[s];
        if (am == 0) {
          z[g][s] = av0;
        } else {
          const int sg = so.sgn[s];
          const float ez = xor_sign(sn[g][am], zmask);
          const float e = sg > 0 ? ez : (sg < 0 ? -ez : xor_sign(ez, qmask));
          z[g][s] = fmaf(cs[g][am], av0, e * bv0);
        }
      }
    }
    float* out = reinterpret_cast<float*>(a.out) + (size_t)(cur.first - a.pair0) * (MH * 256) + 4 * lane;
    V4 acc[G][2];
    float v[G][4];
    for_pieces(std::make_integer_sequence<int, NU>{}, [&](auto uc) __attribute__((always_inline)) {
      constexpr int u = decltype(uc)::value;
      constexpr int sl = u % kSlices, s4 = (u / kSlices) % N4, ti = u / (kSlices * N4);
      // the next unit's pairs once its entry is there, its input once they are
      if (u == vol_stage(NU, NB, 1)) walk.fetch();
      if (u == vol_stage(NU, NB, 2)) {
        nxt = walk.unit();
#pragma unroll
        for (int g = 0; g < G; ++g) rec[g] = recs[nxt.first + (g < nxt.pairs ? g : 0)];
      }
      if (u == vol_stage(NU, NB, 3)) {
#pragma unroll
        for (int g = 0; g < G; ++g) load_x(rec[g], xc[g]);
      }
      f32x4_t(&b)[4] = buf[u % NB];
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const float w = wt[g][4 * sl + t];
          const f32x4_t c = b[t];
#pragma unroll
          for (int j = 0; j < 4; ++j) v[g][j] = sl == 0 && t == 0 ? w * c[j] : fmaf(w, c[j], v[g][j]);
        }
      if (u + NB < NU)
        load_piece(cur.row, u + NB, b);
      else
        load_piece(nxt.row, u + NB - NU, b);
      __builtin_amdgcn_sched_barrier(0);  // (the loads stay here, ahead of what follows)
      if (sl < kSlices - 1) return;
#pragma unroll
      for (int g = 0; g < G; ++g) {
        if (s4 == 0) acc[g][ti & 1] = V4{0, 0, 0, 0};
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[g][ti & 1] = Mfma<float>::op(v[g][j], z[g][4 * s4 + j], acc[g][ti & 1]);
      }
      if (s4 < N4 - 1 || (ti & 1) == 0) return;
      // y (rhs, re|im) of rows 16 i + 4 q + r, rotated by e^{-i m1 phi}
      constexpr int i = ti >> 1;
      for_pieces(std::make_integer_sequence<int, G>{}, [&](auto gc) __attribute__((always_inline)) {
        constexpr int g = decltype(gc)::value;
        float er, ei;
        unsigned mlo, mhi;
        row_phase<LMAX, MMAX, i>(q, hq, cs[g], sn[g], er, ei, mlo, mhi);
        const float elo = xor_sign(ei, mlo), ehi = xor_sign(ei, mhi);
        f32x4_t y;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float eps = r < 2 ? elo : ehi;
          const float al = acc[g][0][r], be = acc[g][1][r];
          const float own = fmaf(al, er, be * eps);
          const float snd = fmaf(be, er, -(al * eps));
          y[r] = fma_xor1(own, sgnz, snd);
        }
        if (g < cur.pairs) *reinterpret_cast<f32x4_t*>(out + (g * MH + i) * 256) = y;
      });
    });
  }
}

// ---- FP64 -------------------------------------------------------------------
// TAP32 (tables of plain FP32 values: no spline moments): the taps come from
// the FP32 kernel's rows (the same values exactly) and are widened in
// registers, half the bytes of the FP64 rows. A piece is four (TAP32) or two
// K-steps of one tile for the four taps of one slice (16 registers). One pair
// at a time: the FP64 products bound it.
template <int LMAX, int MMAX, bool TAP32>
__global__ void __launch_bounds__(kVolThreads, 2) vol_slots64_kernel(VolKArgs a) {
  using Sh = SlotShape<LMAX, MMAX, 4>;
  constexpr int S = Sh::S, NS = Sh::NS, MT = Sh::MT, MH = Sh::MH;
  constexpr int KB = kBatchRhs, KP = TAP32 ? 4 : 2, NP = NS / KP;
  constexpr int NU = MT * NP * kSlices, NB = ring_size(NU, kVolRing64);
  static_assert(KB * 2 == 16, "16 result columns = kBatch right-hand sides x (re, im)");
  static_assert(NS % KP == 0, "whole groups of K-steps");
  static_assert(MMAX <= 4, "phase selection covers |m| <= 4");
  constexpr SlotOrder<LMAX, MMAX> so{};
  static_assert(so.ok, "slot order");
  using Rec = PairRec2<double>;
  using V4 = typename Mfma<double>::v4;
  using TapV = typename std::conditional<TAP32, f32x4_t, f64x2_t>::type;

  const int lane = threadIdx.x & 63;
  const Rec* recs = reinterpret_cast<const Rec*>(a.recs);
  const double* xg = reinterpret_cast<const double*>(a.x);

  const int rr = lane & 15, q = lane >> 4;
  const int rhs = rr >> 1, zp = rr & 1;
  const unsigned zmask = zp ? 0u : 0x80000000u;
  const unsigned qmask = q >= 2 ? 0x80000000u : 0u;
  const double sgnz = zp ? 1.0 : -1.0;
  // the lane's first operand is Re x (re column) or Im x (im column)
  const int64_t xlane = (int64_t)(q * KB + rhs) * NS * 2 + zp, xother = 1 - 2 * zp;

  const unsigned lane16 = 16u * (unsigned)lane;
  TapV buf[NB][4];
  GlobalBytes rows[kSlices][4];
  auto load_piece = [&](int row, int u, TapV (&b)[4]) __attribute__((always_inline)) {
    const int sl = u % kSlices, kp = (u / kSlices) % NP, ti = u / (kSlices * NP);
    const int tile = (ti >> 1) + (ti & 1) * MH;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      if (u < kSlices) rows[sl][t] = vol_row(a.tt, row + vol_tap_offset(a.vmode, sl, t, a.len_z), MT * NP * 1024);
      b[t] = vol_load<TapV>(rows[sl][t], lane16, (tile * NP + kp) * 1024);
    }
  };
  auto load_x = [&](const Rec& r, double (&xs)[2 * NS]) {
    const double* xp = xg + (int64_t)(r.ij & kPairMask) * S * KB * 2 + xlane;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      xs[2 * s] = xp[2 * s];
      xs[2 * s + 1] = xp[2 * s + xother];
    }
  };

  VolWalk walk(a.units, a.bounds);
  VolUnit cur, nxt;
  double xc[2 * NS];
  walk.fetch();
  nxt = walk.unit();
  if (nxt.pairs <= 0) return;
  Rec rec = recs[nxt.first];
#pragma unroll
  for (int u = 0; u < NB; ++u) load_piece(nxt.row, u, buf[u]);
  load_x(rec, xc);

  for (;;) {
    cur = nxt;
    if (cur.pairs <= 0) break;
    double cs[MMAX + 1], sn[MMAX + 1], z[NS], wt[kSlices * 4];
    const double wl = vol_lane_weight<double>(a.vmode, lane, rec.w, rec.w2);
#pragma unroll
    for (int k = 0; k < kSlices * 4; ++k) wt[k] = lane_value(wl, k);
    phase_powers64<MMAX>(rec.c, rec.s, cs, sn);
    // B operand per K-step: (e^{i m2 phi} x[slot 4 s + q][rhs]).re or .im
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const int am = so.absm[s];
      const double av = xc[2 * s], bv = xc[2 * s + 1];
      if (am == 0) {
        z[s] = av;
      } else {
        const int sg = so.sgn[s];
        const double ez = xor_sign64(sn[am], zmask);
        const double ee = sg > 0 ? ez : (sg < 0 ? -ez : xor_sign64(ez, qmask));
        z[s] = fma(cs[am], av, ee * bv);
      }
    }
    double* out = reinterpret_cast<double*>(a.out) + (size_t)(cur.first - a.pair0) * (MH * 256) + lane;
    V4 acc[2];
    double v[KP];
    for_pieces(std::make_integer_sequence<int, NU>{}, [&](auto uc) __attribute__((always_inline)) {
      constexpr int u = decltype(uc)::value;
      constexpr int sl = u % kSlices, kp = (u / kSlices) % NP, ti = u / (kSlices * NP);
      if (u == vol_stage(NU, NB, 1)) walk.fetch();
      if (u == vol_stage(NU, NB, 2)) {
        nxt = walk.unit();
        rec = recs[nxt.first];
      }
      if (u == vol_stage(NU, NB, 3)) load_x(rec, xc);
      TapV(&b)[4] = buf[u % NB];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const double w = wt[4 * sl + t];
#pragma unroll
        for (int j = 0; j < KP; ++j) {
          const double c = (double)b[t][j];
          v[j] = sl == 0 && t == 0 ? w * c : fma(w, c, v[j]);
        }
      }
      if (u + NB < NU)
        load_piece(cur.row, u + NB, b);
      else
        load_piece(nxt.row, u + NB - NU, b);
      __builtin_amdgcn_sched_barrier(0);
      if (sl < kSlices - 1) return;
      if (kp == 0) acc[ti & 1] = V4{0, 0, 0, 0};
#pragma unroll
      for (int j = 0; j < KP; ++j) acc[ti & 1] = Mfma<double>::op(v[j], z[KP * kp + j], acc[ti & 1]);
      if (kp < NP - 1 || (ti & 1) == 0) return;
      // register r of tile i: slot 16 i + 4 r + q (group 4 i + r), rotated by e^{-i m1 phi}
      constexpr int i = ti >> 1;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int g = 4 * i + r;
        const int am = so.absm[g], sg = so.sgn[g];
        const double er = cs[am];
        const double eps = am == 0 ? 0.0 : (sg > 0 ? sn[am] : (sg < 0 ? -sn[am] : xor_sign64(sn[am], qmask)));
        const double al = acc[0][r], be = acc[1][r];
        const double own = fma(al, er, be * eps);
        const double snd = fma(be, er, -(al * eps));
        out[(i * 4 + r) * 64] = fma(sgnz, lane_xor1_64(snd), own);
      }
    });
  }
}

// ---- FP16 operands ----------------------------------------------------------
// The table holds each tap row divided by its own power of two hscale[row]; a
// pair's taps are weighted with vol_tap_weight hscale[row] / (the largest of
// the entry's scales), which then scales the result. A piece is one tap row.
template <int LMAX, int MMAX>
__global__ void __launch_bounds__(kVolThreads, 2) vol_half_kernel(VolKArgs a) {
  using Sh = SlotShape<LMAX, MMAX, 4>;
  constexpr int S = Sh::S, MT = Sh::MT, MH = Sh::MH;
  constexpr int NC = S / 16, KB = kBatchRhs, G = kVolPairs32;
  constexpr int NU = 4 * kSlices, NB = ring_size(NU, NC <= 2 ? kVolRingHalf : 2);
  static_assert(KB * 2 == 16, "16 result columns = kBatch right-hand sides x (re, im)");
  static_assert(S % 16 == 0 && MH == NC, "result tile c and input chunk c share the lane's slot group");
  constexpr SlotOrder<LMAX, MMAX> so{};
  static_assert(so.ok, "slot order");
  using Rec = PairRec2<float>;
  using V4 = typename Mfma<float>::v4;

  const float xmax = *a.xmax;
  const int lane = threadIdx.x & 63;
  const Rec* recs = reinterpret_cast<const Rec*>(a.recs);
  const _Float16* xg = reinterpret_cast<const _Float16*>(a.x);

  const int rr = lane & 15, q = lane >> 4;
  const int rhs = rr >> 1, zp = rr & 1;
  const float hq[4] = {q == 0 ? 1.f : 0.f, q == 1 ? 1.f : 0.f, q == 2 ? 1.f : 0.f, q == 3 ? 1.f : 0.f};
  // signs: z of the re column takes -b; the im column's receiver rotation -sin; the Lim half
  // of K -Im z (re column) or Re z (im column)
  const unsigned zmask = zp ? 0u : 0x80000000u, ymask = zp ? 0x80000000u : 0u, hsign = zp ? 0u : 0x80008000u;
  const int64_t xlane = (int64_t)(q * KB + rhs) * NC * 8 + 4 * zp, xother = 4 - 8 * zp;
  // tap row of lane 4 s + t relative to the entry's first
  const int tap_off = vol_tap_offset(a.vmode, (lane >> 2) & 3, lane & 3, a.len_z);

  const unsigned lane_off = 8u * NC * (unsigned)lane;
  u32x2_t buf[NB][MT][NC];
  auto load_piece = [&](int row, int u, u32x2_t (&b)[MT][NC]) __attribute__((always_inline)) {
    const GlobalBytes r = vol_row(a.tt, row + vol_tap_offset(a.vmode, u >> 2, u & 3, a.len_z), MT * 64 * NC * 8);
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      if constexpr (NC % 2 == 0) {
#pragma unroll
        for (int c = 0; c < NC; c += 2) {
          const u32x4_t v = vol_load<u32x4_t>(r, lane_off, i * 64 * NC * 8 + 8 * c);
          b[i][c] = u32x2_t{v.x, v.y};
          b[i][c + 1] = u32x2_t{v.z, v.w};
        }
      } else {
#pragma unroll
        for (int c = 0; c < NC; ++c) b[i][c] = vol_load<u32x2_t>(r, lane_off, i * 64 * NC * 8 + 8 * c);
      }
    }
  };
  auto load_x = [&](const Rec& r, uint2 (&xs)[2 * NC]) {
    const _Float16* xp = xg + (int64_t)(r.ij & kPairMask) * S * KB * 2 + xlane;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      xs[2 * c] = *reinterpret_cast<const uint2*>(xp + 8 * c);
      xs[2 * c + 1] = *reinterpret_cast<const uint2*>(xp + 8 * c + xother);
    }
  };

  VolWalk walk(a.units, a.bounds);
  VolUnit cur, nxt;
  Rec rec[G];
  uint2 xc[G][2 * NC];
  walk.fetch();
  nxt = walk.unit();
  if (nxt.pairs <= 0) return;
#pragma unroll
  for (int g = 0; g < G; ++g) rec[g] = recs[nxt.first + (g < nxt.pairs ? g : 0)];
  float hs = a.hscale[nxt.row + tap_off];
#pragma unroll
  for (int u = 0; u < NB; ++u) load_piece(nxt.row, u, buf[u]);
#pragma unroll
  for (int g = 0; g < G; ++g) load_x(rec[g], xc[g]);

  for (;;) {
    cur = nxt;
    if (cur.pairs <= 0) break;
    // the weights relative to the largest of the entry's scales (powers of two: exact)
    float hmax = hs;
#pragma unroll
    for (int k = 1; k < 4 * kSlices; k *= 2) hmax = fmaxf(hmax, __shfl_xor(hmax, k));
    const float scl = hmax * xmax, rel = hs / hmax;
    half2_t wl[G];
    float cs[G][MMAX + 1], sn[G][MMAX + 1];
    half4_t zb[G][NC], zb2[G][NC];
    for_pieces(std::make_integer_sequence<int, G>{}, [&](auto gc) __attribute__((always_inline)) {
      constexpr int g = decltype(gc)::value;
      const _Float16 wh =
          (_Float16)(vol_lane_weight<float>(a.vmode, lane, rec[g].w, rec[g].w2) * rel);
      wl[g] = half2_t{wh, wh};
      phase_powers<MMAX>(rec[g].c, rec[g].s, cs[g], sn[g]);
      for_pieces(std::make_integer_sequence<int, NC>{}, [&](auto cc) __attribute__((always_inline)) {
        constexpr int c = decltype(cc)::value;
        float cz, sz;
        unsigned mlo, mhi;
        row_phase<LMAX, MMAX, c>(q, hq, cs[g], sn[g], cz, sz, mlo, mhi);
        // zb: the lane's column of z = e^{i m2 phi} x; zb2: the column of the other part with
        // the sign of the complex product
        const _Float16 czh = (_Float16)cz;
        const _Float16 eloh = (_Float16)xor_sign(sz, mlo ^ zmask), ehih = (_Float16)xor_sign(sz, mhi ^ zmask);
        const half2_t cz2 = {czh, czh}, elo2 = {eloh, eloh}, ehi2 = {ehih, ehih};
        const half2_t a01 = __builtin_bit_cast(half2_t, xc[g][2 * c].x), a23 = __builtin_bit_cast(half2_t, xc[g][2 * c].y);
        const half2_t b01 = __builtin_bit_cast(half2_t, xc[g][2 * c + 1].x);
        const half2_t b23 = __builtin_bit_cast(half2_t, xc[g][2 * c + 1].y);
        const half2_t z01 = a01 * cz2 + b01 * elo2, z23 = a23 * cz2 + b23 * ehi2;
        zb[g][c] = half4_t{z01[0], z01[1], z23[0], z23[1]};
        const half2_t y01 = b01 * cz2 - a01 * elo2, y23 = b23 * cz2 - a23 * ehi2;
        zb2[g][c] =
            __builtin_bit_cast(half4_t, __builtin_bit_cast(u32x2_t, half4_t{y01[0], y01[1], y23[0], y23[1]}) ^ hsign);
      });
    });
    float* out = reinterpret_cast<float*>(a.out) + (size_t)(cur.first - a.pair0) * (MH * 256) + 4 * lane;

    V4 acc[G][MH];
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int i = 0; i < MH; ++i) acc[g][i] = V4{0, 0, 0, 0};
    for_pieces(std::make_integer_sequence<int, NU>{}, [&](auto uc) __attribute__((always_inline)) {
      constexpr int u = decltype(uc)::value;
      if (u == vol_stage(NU, NB, 1)) walk.fetch();
      if (u == vol_stage(NU, NB, 2)) {
        nxt = walk.unit();
#pragma unroll
        for (int g = 0; g < G; ++g) rec[g] = recs[nxt.first + (g < nxt.pairs ? g : 0)];
        hs = a.hscale[nxt.row + tap_off];
      }
      if (u == vol_stage(NU, NB, 3)) {
#pragma unroll
        for (int g = 0; g < G; ++g) load_x(rec[g], xc[g]);
      }
      u32x2_t(&b)[MT][NC] = buf[u % NB];
      // one 16x16x32 MFMA per row tile and chunk: the lane's 8 K values are its 4 slots of the
      // chunk from Re L (times zb) and the same 4 from Im L (times zb2)
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const half2_t wt = __builtin_bit_cast(half2_t, __builtin_amdgcn_readlane(__builtin_bit_cast(int, wl[g]), u));
        const half4_t wt4 = {wt[0], wt[1], wt[0], wt[1]};
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          const half8_t bv = __builtin_shufflevector(zb[g][c] * wt4, zb2[g][c] * wt4, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
          for (int i = 0; i < MH; ++i) {
            const half4_t re = __builtin_bit_cast(half4_t, b[i][c]), im = __builtin_bit_cast(half4_t, b[i + MH][c]);
            const half8_t av = __builtin_shufflevector(re, im, 0, 1, 2, 3, 4, 5, 6, 7);
            acc[g][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av, bv, acc[g][i], 0, 0, 0);
          }
        }
      }
      if (u + NB < NU)
        load_piece(cur.row, u + NB, b);
      else
        load_piece(nxt.row, u + NB - NU, b);
      __builtin_amdgcn_sched_barrier(0);
    });
    // y (rhs, re|im) of rows 16 i + 4 q + r, rotated by e^{-i m1 phi}, times the operand scales
    for_pieces(std::make_integer_sequence<int, G * MH>{}, [&](auto gi) __attribute__((always_inline)) {
        constexpr int g = decltype(gi)::value / MH, i = decltype(gi)::value % MH;
        float er, ei;
        unsigned mlo, mhi;
        row_phase<LMAX, MMAX, i>(q, hq, cs[g], sn[g], er, ei, mlo, mhi);
        er *= scl;
        ei *= scl;
        // (the im column takes -sin: y'_im = cos y_im - sin y_re)
        const float elo = xor_sign(ei, mlo ^ ymask), ehi = xor_sign(ei, mhi ^ ymask);
        f32x4_t y;
#pragma unroll
        for (int r = 0; r < 4; ++r) y[r] = fmaf(er, acc[g][i][r], (r < 2 ? elo : ehi) * lane_xor1(acc[g][i][r]));
        if (g < cur.pairs) *reinterpret_cast<f32x4_t*>(out + (g * MH + i) * 256) = y;
      });
  }
}

}  // namespace smh
