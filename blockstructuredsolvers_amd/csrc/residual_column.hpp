// residual_column.hpp -- FP64 residual of one right-hand side, a wave per block row.
#pragma once

#include <type_traits>

#include "common.hpp"
#include "mixed.hpp"

namespace bss {

constexpr int kParts = 64;      // partial maxima of a work item: [0,16) max|r_j|,
constexpr int kMnormSlot = 48;  // [16,32) max|x_j|, [32,48) max|d_j|, [48] max row sum of |M|

// NaN-propagating max (fmax would drop a NaN residual and report convergence)
__device__ inline double nmax(double a, double b) { return (b > a || b != b) ? b : a; }

// x[lane] from another lane of the same 16 (DPP control CTRL)
template <int CTRL>
__device__ inline double dpp64(double x) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(x), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(x), CTRL, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}
constexpr int kDppXor1 = 0xB1, kDppXor2 = 0x4E, kDppHalfMirror = 0x141, kDppRor8 = 0x128;

// How a wave holds an NB x NB block: a lane has two consecutive rows (16 bytes), R lanes a
// column, and load j of NI reads column g NI + j in lane group g.
template <int NB>
struct ColMap {
  static constexpr int R = NB / 2;
  static constexpr int CPI = 64 / R;         // columns a load reads
  static constexpr int NI = NB / CPI;        // loads of a block
  static constexpr int G = NI < 8 ? NI : 8;  // loads of a chunk
  static constexpr int NC = NI / G;
  // lanes whose values one column sum folds, and the sums a column is left with
  static constexpr int FOLD = R == 64 ? 64 : R == 32 ? 32 : R % 16 == 0 ? 16 : 8;
  static constexpr int P = R / FOLD;
  static_assert(NI * CPI == NB && G * NC == NI && (G == 8 || G == 2), "chunks");
  static_assert(NC % 2 == 0 || NC <= 3, "chunks alternate between two buffers");

  // Sum over FOLD lanes of the G values of each lane; on return the lane holds value
  // slot(l).  Each step of a halving sends the half a lane gives up to its partner: the
  // partners are the lanes of one octet (half mirror, then lanes l ^ 2 and l ^ 1).
  __device__ static inline int slot(int l) { return G == 8 ? l & 7 : (l >> 2) & 1; }
  template <int CTRL, int N>
  __device__ static inline void halve(double (&v)[G], bool up) {
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const double keep = up ? v[N + j] : v[j], send = up ? v[j] : v[N + j];
      v[j] = keep + dpp64<CTRL>(send);
    }
  }
  __device__ static inline double fold(double (&v)[G], int l) {
    halve<kDppHalfMirror, G / 2>(v, (l & 4) != 0);
    if constexpr (G == 8) {
      halve<kDppXor2, 2>(v, (l & 2) != 0);
      halve<kDppXor1, 1>(v, (l & 1) != 0);
    } else {
      v[0] += dpp64<kDppXor2>(v[0]);
      v[0] += dpp64<kDppXor1>(v[0]);
    }
    double t = v[0];
    if constexpr (FOLD >= 16) t += dpp64<kDppRor8>(t);
    if constexpr (FOLD == 64) t = row4_sum(t);
    if constexpr (FOLD == 32) {
      const unsigned lo = (unsigned)__double2loint(t), hi = (unsigned)__double2hiint(t);
      const auto rl = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
      const auto rh = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
      t = __hiloint2double((int)rh[0], (int)rl[0]) + __hiloint2double((int)rh[1], (int)rl[1]);
    }
    return t;
  }
};

constexpr int kColWaves = 4;  // waves of a work-group: block rows of an item in flight

// Residual pass over one work item (a block range [b0, b1) of one system), one right-hand
// side:
//   x_new = x_old + dx (FP64; written for the item's own blocks),
//   r = d - (B_{i-1}^T x_{i-1} + A_i x_i + B_i x_{i+1}) in FP64, stored as FP32 for the
//   next correction solve, plus max |r|, |x|, |d|, and (MN) the largest row sum of |M|.
// HBM-bound.  The item's block rows are split over the waves, and a wave does its rows
// alone: two chunks of eight 16-byte loads a lane in turn, one in flight while the other
// is used, so nothing waits at a barrier and sixteen waves keep 128 KB a CU in flight.
// Every block is read once and only A's upper triangle: a lane below the diagonal repeats
// the column's last upper rows (same cache lines) and drops them.  A value serves both its
// row (a running sum of the lane) and its column (products folded over the lanes: B_i^T
// x_i goes to row i + 1, the strict upper part of A_i to row i itself).  The wave that owns
// row i + 1 gets the carry of row i through LDS at the end; the carry into the item is one
// more pass over B_{b0-1} by the last wave, whose share is never the largest.
// Measured against a work-group per block row with A read whole (a barrier pair a row): 32
// systems of 8192 blocks, n = 64: 3.44 -> 2.69 ms (14.0 GB, 5.2 TB/s), with ||M|| 3.50 ->
// 2.69; 8 systems of 2048 blocks, n = 96: 0.50 -> 0.37 ms, with ||M|| 0.53 -> 0.38.
// Eight waves a work-group at 128 registers spill; four at 168 give the same bytes in
// flight.
// X0: x_old is zero (the first pass of a solve), and neither read nor there.
template <int NB, bool MN, bool X0>
__global__ void __launch_bounds__(64 * kColWaves)
    __attribute__((amdgpu_waves_per_eu(NB == 96 && MN ? 2 : 3)))  // (LDS: two work-groups a CU)
    residual_column_kernel(const ResItem* __restrict__ items, const ResSys* __restrict__ systems,
                           double* __restrict__ part, int xo_k, int dx_k, int xn_k, int ro_k) {
  typedef ColMap<NB> M;
  constexpr int R = M::R, CPI = M::CPI, NI = M::NI, G = M::G, NC = M::NC, P = M::P;
  constexpr int KW = kColWaves, K2 = MN ? 2 : 1;
  constexpr int PD = P + (R * CPI < 64 ? 1 : 0);  // and a place for the sums to drop
  constexpr long long NN = (long long)NB * NB;
  // two doubles or floats of consecutive rows: 8 or 4 bytes of alignment is all the
  // caller's buffers promise
  typedef double d2_t __attribute__((ext_vector_type(2), aligned(8)));
  typedef float f2_t __attribute__((ext_vector_type(2), aligned(4)));
  typedef double l2_t __attribute__((ext_vector_type(2)));

  __shared__ __attribute__((aligned(16))) double Xw[KW][2][NB];         // x of rows i, i + 1
  __shared__ __attribute__((aligned(16))) double Tw[KW][2 * K2][PD][NB];  // column sums: B, A
  __shared__ __attribute__((aligned(16))) double Yw[KW][K2][CPI > 1 ? CPI : 1][CPI > 1 ? NB : 2];
  __shared__ __attribute__((aligned(16))) double Cw[KW + 1][K2][NB];    // carries
  __shared__ __attribute__((aligned(16))) double Fw[KW][K2][NB];        // first rows, no carry
  __shared__ double red[KW][4];

  const ResItem it = items[blockIdx.x];
  const ResSys& S = systems[it.sys];
  const int N = S.N, b0 = it.b0, b1 = it.b1;
  const int w = wave_id(), l = lane_id();
  // this lane's column group and row pair; the lanes left over (n = 48 and 96) repeat the
  // last pair and their column sums are dropped
  const bool act = l < R * CPI;
  const int g = act ? l / R : CPI - 1, q = act ? l % R : R - 1;
  const int pl = act ? l % R / M::FOLD : P;  // this lane's column sums go here
  const int hk = q - g * (NI / 2);  // row pair against column pair
  const auto As = gptr((const double*)S.A);
  const auto Bs = gptr((const double*)S.B);
  const auto ds = gptr((const double*)S.d);
  const auto xo = gptr((const double*)(X0 ? nullptr : S.x[xo_k]));
  const auto dxs = gptr((const float*)S.v[dx_k]);
  const auto xn = gptr(S.x[xn_k]);
  const auto ro = gptr(S.v[ro_k]);
  auto fence = [] {  // LDS of one wave: orders the compiler, the hardware is in order
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };

  struct xv_t {
    d2_t o;
    f2_t d;
  };
  auto load_x = [&](int j) -> xv_t {  // clamped: every load is unconditional
    const long long e = (long long)(j < 0 ? 0 : j >= N ? N - 1 : j) * NB + 2 * q;
    const f2_t d = *(const BSS_GLOBAL f2_t*)(dxs + e);
    if constexpr (X0) return xv_t{d2_t{0.0, 0.0}, d};
    else return xv_t{*(const BSS_GLOBAL d2_t*)(xo + e), d};
  };
  auto sum_x = [&](const xv_t& v, int j) -> l2_t {
    const bool in = j >= 0 && j < N;
    const double x0 = v.o[0] + (double)v.d[0], x1 = v.o[1] + (double)v.d[1];
    return l2_t{in ? x0 : 0.0, in ? x1 : 0.0};
  };
  auto put_x = [&](int j, const l2_t& x) { *(l2_t*)&Xw[w][j & 1][2 * q] = x; };

  // chunk c of a block: full (base + lane offset), or its upper triangle.  The offsets are
  // made opaque where they are used: kept over the loop for every load they would spill.
  const int lcol = g * NI * NB + 2 * q;
  auto load_full = [&](d2_t(&u)[G], const BSS_GLOBAL double* b, int c) {
    unsigned o = 8 * lcol;
    asm volatile("" : "+v"(o));
#pragma unroll
    for (int j = 0; j < G; ++j)
      u[j] = *(const BSS_GLOBAL d2_t*)((const BSS_GLOBAL char*)(b + (c * G + j) * NB) + o);
  };
  auto load_upper = [&](d2_t(&u)[G], const BSS_GLOBAL double* a, int c) {
    int k0 = g * NI + c * G;
    asm volatile("" : "+v"(k0));
#pragma unroll
    for (int j = 0; j < G; ++j) {
      const unsigned o = 8 * (k0 * NB + min(2 * q, k0 + (j & ~1)));
      u[j] = *(const BSS_GLOBAL d2_t*)((const BSS_GLOBAL char*)(a + j * NB) + o);
    }
  };
  double y0 = 0, y1 = 0, s0 = 0, s1 = 0;  // this lane's rows: M x and row sums of |M|
  // column sums of chunk c to LDS
  auto put_sum = [&](double(&t)[G], int k2, int c) {
    const double v = M::fold(t, l);
    Tw[w][k2][pl][g * NI + c * G + M::slot(l)] = v;
  };
  // column sums of this lane's rows
  auto get_sum = [&](int k2) -> l2_t {
    l2_t t = *(const l2_t*)&Tw[w][k2][0][2 * q];
#pragma unroll
    for (int p = 1; p < P; ++p) t += *(const l2_t*)&Tw[w][k2][p][2 * q];
    return t;
  };
  // B's chunk c: B x_{i+1} to the rows (Y), B^T x_i to the columns
  auto use_b = [&](const d2_t(&u)[G], int c, const double* xc, const l2_t& xr, auto with_y) {
    double t[G];
#pragma unroll
    for (int j = 0; j < G; ++j) {
      if constexpr (decltype(with_y)::value) {
        const double xk = xc[g * NI + c * G + j];
        y0 = fma(u[j][0], xk, y0);
        y1 = fma(u[j][1], xk, y1);
      }
      t[j] = fma(u[j][1], xr[1], u[j][0] * xr[0]);
    }
    put_sum(t, 0, c);
    if constexpr (MN) {
#pragma unroll
      for (int j = 0; j < G; ++j) {
        if constexpr (decltype(with_y)::value) {
          s0 += fabs(u[j][0]);
          s1 += fabs(u[j][1]);
        }
        t[j] = fabs(u[j][0]) + fabs(u[j][1]);
      }
      put_sum(t, 2, c);
    }
  };
  // A's chunk c: rows 2q and 2q + 1 of column k = g NI + c G + j are in the upper triangle
  // where they are at most k, and give to row k where they are less
  auto use_a = [&](const d2_t(&u)[G], int c, const double* xc, const l2_t& xr) {
    double t[G], ta[G];
    int h = hk - c * (G / 2);
    asm volatile("" : "+v"(h));
#pragma unroll
    for (int j = 0; j < G; ++j) {
      const bool at = h <= j / 2, below = h < j / 2;
      const double u0 = at ? u[j][0] : 0.0;
      const double u1 = (j & 1 ? at : below) ? u[j][1] : 0.0;
      const double v0 = j & 1 ? u0 : (below ? u[j][0] : 0.0);
      const double v1 = j & 1 ? (below ? u[j][1] : 0.0) : u1;
      const double xk = xc[g * NI + c * G + j];
      y0 = fma(u0, xk, y0);
      y1 = fma(u1, xk, y1);
      t[j] = fma(v1, xr[1], v0 * xr[0]);
      if constexpr (MN) {
        s0 += fabs(u0);
        s1 += fabs(u1);
        ta[j] = fabs(v0) + fabs(v1);
      }
    }
    put_sum(t, 1, c);
    if constexpr (MN) put_sum(ta, 3, c);
  };
  // a lane's row sums over its columns, added up over the column groups
  auto row_sums = [&](int k2, double a, double b) -> l2_t {
    if constexpr (CPI == 1) return l2_t{a, b};
    *(l2_t*)&Yw[w][k2][g][2 * q] = l2_t{a, b};
    fence();
    l2_t y = *(const l2_t*)&Yw[w][k2][0][2 * q];
#pragma unroll
    for (int p = 1; p < CPI; ++p) y += *(const l2_t*)&Yw[w][k2][p][2 * q];
    fence();
    return y;
  };
  const int per = (b1 - b0 + KW - 1) / KW;
  const int w0 = b0 + w * per, w1 = min(w0 + per, b1);
  d2_t ua[G], ub[G];

  // the carry into the item's first row
  if (w == KW - 1) {
    l2_t t = {0.0, 0.0}, ta = {0.0, 0.0};
    if (b0 > 0) {
      const l2_t x = sum_x(load_x(b0 - 1), b0 - 1);
      const auto Bb = Bs + (b0 - 1) * NN;
#pragma unroll 1
      for (int c = 0; c < NC; ++c) {
        load_full(ua, Bb, c);
        use_b(ua, c, nullptr, x, std::false_type());
      }
      fence();
      t = get_sum(0);
      if constexpr (MN) ta = get_sum(2);
      fence();
    }
    *(l2_t*)&Cw[0][0][2 * q] = t;
    if constexpr (MN) *(l2_t*)&Cw[0][1][2 * q] = ta;
  }

  double rmax = 0.0, xmax = 0.0, dmax = 0.0, mmax = 0.0;
  auto finish = [&](long long blk, const l2_t& r, const l2_t& s) {
    *(BSS_GLOBAL f2_t*)(ro + blk * NB + 2 * q) = f2_t{(float)r[0], (float)r[1]};
    rmax = nmax(rmax, nmax(fabs(r[0]), fabs(r[1])));
    if constexpr (MN) mmax = nmax(mmax, nmax(s[0], s[1]));
  };
  if (w0 < w1) {
    // A row's coupling; the system's last row has none, and reads its A in its place
    auto b_base = [&](int i) { return i + 1 < N ? Bs + i * NN : As + i * NN; };
    const xv_t xa = load_x(w0), xb = load_x(w0 + 1);
    load_full(ua, b_base(w0), 0);
    l2_t x0 = sum_x(xa, w0);
    put_x(w0, x0);
    put_x(w0 + 1, sum_x(xb, w0 + 1));
    // Cw[w + 1]: the carry into the row at hand; the wave's first row goes without
    *(l2_t*)&Cw[w + 1][0][2 * q] = l2_t{0.0, 0.0};
    if constexpr (MN) *(l2_t*)&Cw[w + 1][1][2 * q] = l2_t{0.0, 0.0};
    fence();
#pragma unroll 1
    for (int i = w0; i < w1; ++i) {
      const bool next = i + 1 < N, more = i + 1 < w1;
      const auto Ab = As + i * NN, Bb = b_base(i);
      // next row's first chunk; after the wave's last row something at hand
      const auto Bn = more ? b_base(i + 1) : Ab + (long long)(NC - 1) * G * NB;
      const double *xi = Xw[w][i & 1], *xp = Xw[w][(i + 1) & 1];
      const xv_t xq = load_x(i + 2);
      const d2_t dv = *(const BSS_GLOBAL d2_t*)(ds + (long long)i * NB + 2 * q);
      y0 = y1 = s0 = s1 = 0.0;
      auto do_b = [&](const d2_t(&u)[G], int c) {
        if (next) use_b(u, c, xp, x0, std::true_type());
      };
      auto do_a = [&](const d2_t(&u)[G], int c) { use_a(u, c, xi, x0); };
      auto order = [] { __builtin_amdgcn_sched_barrier(0); };
      if constexpr (NC % 2 == 0) {
#pragma unroll 1
        for (int c = 0; c + 2 < NC; c += 2) {
          load_full(ub, Bb, c + 1);
          order();
          do_b(ua, c);
          load_full(ua, Bb, c + 2);
          order();
          do_b(ub, c + 1);
        }
        load_full(ub, Bb, NC - 1);
        order();
        do_b(ua, NC - 2);
        load_upper(ua, Ab, 0);
        order();
        do_b(ub, NC - 1);
#pragma unroll 1
        for (int c = 0; c + 2 < NC; c += 2) {
          load_upper(ub, Ab, c + 1);
          order();
          do_a(ua, c);
          load_upper(ua, Ab, c + 2);
          order();
          do_a(ub, c + 1);
        }
        load_upper(ub, Ab, NC - 1);
        order();
        do_a(ua, NC - 2);
        load_full(ua, Bn, 0);
        order();
        do_a(ub, NC - 1);
      } else if constexpr (NC == 3) {
        load_full(ub, Bb, 1);
        order();
        do_b(ua, 0);
        load_full(ua, Bb, 2);
        order();
        do_b(ub, 1);
        load_upper(ub, Ab, 0);
        order();
        do_b(ua, 2);
        load_upper(ua, Ab, 1);
        order();
        do_a(ub, 0);
        load_upper(ub, Ab, 2);
        order();
        do_a(ua, 1);
        load_full(ua, Bn, 0);
        order();
        do_a(ub, 2);
      } else {
        load_upper(ub, Ab, 0);
        order();
        do_b(ua, 0);
        load_full(ua, Bn, 0);
        order();
        do_a(ub, 0);
      }
      fence();
      // r_i = d_i - (carry + rows of A and B + the strict upper part of A transposed)
      const l2_t y = row_sums(0, y0, y1) + get_sum(1) + *(const l2_t*)&Cw[w + 1][0][2 * q];
      const l2_t r = {dv[0] - y[0], dv[1] - y[1]};
      l2_t s = {0.0, 0.0};
      if constexpr (MN) s = row_sums(1, s0, s1) + get_sum(3) + *(const l2_t*)&Cw[w + 1][1][2 * q];
      *(BSS_GLOBAL d2_t*)(xn + (long long)i * NB + 2 * q) = d2_t{x0[0], x0[1]};
      xmax = nmax(xmax, nmax(fabs(x0[0]), fabs(x0[1])));
      dmax = nmax(dmax, nmax(fabs(dv[0]), fabs(dv[1])));
      if (i == w0) {
        *(l2_t*)&Fw[w][0][2 * q] = r;
        if constexpr (MN) *(l2_t*)&Fw[w][1][2 * q] = s;
      } else {
        finish(i, r, s);
      }
      // the carry into row i + 1 (the system's last row has none, and no sums)
      l2_t t = get_sum(0);
      if (!next) t = l2_t{0.0, 0.0};
      if constexpr (MN) s = get_sum(2);
      if (!next) s = l2_t{0.0, 0.0};
      fence();
      *(l2_t*)&Cw[w + 1][0][2 * q] = t;
      if constexpr (MN) *(l2_t*)&Cw[w + 1][1][2 * q] = s;
      x0 = *(const l2_t*)&xp[2 * q];
      put_x(i + 2, sum_x(xq, i + 2));
      fence();
    }
  }
  __syncthreads();
  if (w0 < w1) {
    const l2_t c = *(const l2_t*)&Cw[w][0][2 * q];
    const l2_t r = *(const l2_t*)&Fw[w][0][2 * q] - c;
    l2_t s = {0.0, 0.0};
    if constexpr (MN) s = *(const l2_t*)&Fw[w][1][2 * q] + *(const l2_t*)&Cw[w][1][2 * q];
    finish(w0, r, s);
  }
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    rmax = nmax(rmax, __shfl_xor(rmax, o));
    xmax = nmax(xmax, __shfl_xor(xmax, o));
    dmax = nmax(dmax, __shfl_xor(dmax, o));
    if constexpr (MN) mmax = nmax(mmax, __shfl_xor(mmax, o));
  }
  if (l == 0) {
    red[w][0] = rmax;
    red[w][1] = xmax;
    red[w][2] = dmax;
    red[w][3] = mmax;
  }
  __syncthreads();
  if (threadIdx.x < 4) {
    double m = red[0][threadIdx.x];
    for (int k = 1; k < KW; ++k) m = nmax(m, red[k][threadIdx.x]);
    part[(long long)blockIdx.x * kParts + 16 * threadIdx.x] = m;
  }
}

}  // namespace bss
