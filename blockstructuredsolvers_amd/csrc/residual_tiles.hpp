// residual_tiles.hpp -- FP64 residual of several right-hand sides on MFMA, a wave per
// block row.
#pragma once

#include <type_traits>
#include <utility>

#include "common.hpp"
#include "mixed.hpp"
#include "residual_column.hpp"

namespace bss {

// The tiles of one block row in the order a wave takes them: A's upper tiles, then B's,
// column by column; RING tiles (the most that leave the registers without spills, up to a
// few at n = 64 and 128) are in registers or in flight, and the row is padded to a
// multiple of that, so that a tile has the same registers in every row.
template <int NB, bool MN>
struct RowTiles {
  static constexpr int TT = NB / 16;
  static constexpr int NA = TT * (TT + 1) / 2, T = NA + TT * TT;
  static constexpr int RING = NB == 16   ? 2
                              : NB == 32 ? 4
                              : NB == 48 ? 5
                              : NB == 64 ? (MN ? 4 : 5)
                              : NB == 96 ? 10
                              : MN       ? 5
                                         : 8;
  static constexpr int STEPS = (T + RING - 1) / RING * RING;
  static constexpr bool is_a(int s) { return s < NA; }
  static constexpr int col(int s) {
    if (s >= NA) return (s - NA) / TT;
    int c = 0;
    while ((c + 1) * (c + 2) / 2 <= s) ++c;
    return c;
  }
  static constexpr int row(int s) {
    return s >= NA ? (s - NA) % TT : s - col(s) * (col(s) + 1) / 2;
  }
  // registers: -x of two block rows, two rows of results, the ring
  static constexpr int waves_per_eu() { return NB <= 32 ? 3 : NB <= 64 ? 2 : 1; }
};

template <typename F, int... s>
__device__ __attribute__((always_inline)) inline void for_each_step(
    F& step, std::integer_sequence<int, s...>) {
  (step(std::integral_constant<int, s>{}), ...);
}

// Residual pass over one work item (a block range [b0, b1) of one system), several
// right-hand sides:
//   x_new = x_old + dx (FP64; written for the item's own blocks),
//   r = d - (B_{i-1}^T x_{i-1} + A_i x_i + B_i x_{i+1}) in FP64 on MFMA, stored as FP32
//   for the next correction solve, plus per-column max |r|, |x|, |d|, and (MN) the largest
//   row sum of |M|.
// HBM-bound.  The item's block rows are split over the waves, as in
// residual_column_kernel, and a wave does its rows alone: RING tiles in flight, no
// barrier.  A tile is read once (and only A's upper ones) and serves two products: as
// loaded, lane (row lr, column 4 lk + q) is the B operand of x^T M^T, and through 2 KB of
// LDS, lane (column lr, row 4 lk + q), of x^T M; x lies in registers as the A operand of
// both.  The results have the right-hand side in lk and the row in lr, which is the order
// of d and r in memory.  -x is kept in place of x and the results start from d, so no
// product is negated; the sums that B_i^T x_i starts for row i + 1 become that row's
// results as they are.  The wave's first row waits in LDS for its share of the row before,
// which the wave before adds at the end.
// Measured against a work-group per block row (two barriers a row, B read a second time as
// transposed operand, A read whole), 8 systems of 4096 blocks, n = 64, 16 right-hand sides:
// 712 -> 604 us, 2.8 GB at 4.6 TB/s (a copy reaches 4.9, reads alone 6.1).
// X0: x_old is zero (the first pass of a solve), and neither read nor there.
template <int NB, bool MN, bool X0>
__global__ void __launch_bounds__(64 * kColWaves)
    __attribute__((amdgpu_waves_per_eu(RowTiles<NB, MN>::waves_per_eu())))
    residual_tiles_kernel(const ResItem* __restrict__ items, const ResSys* __restrict__ systems,
                          double* __restrict__ part, int nrhs, int xo_k, int dx_k, int xn_k,
                          int ro_k) {
  typedef RowTiles<NB, MN> RT;
  constexpr int TT = RT::TT, RING = RT::RING, KW = kColWaves, LDT = 18;
  constexpr long long NN = (long long)NB * NB;
  typedef Mfma<double>::acc_t acc_t;
  typedef double d2_t __attribute__((ext_vector_type(2), aligned(8)));
  typedef float f4u_t __attribute__((ext_vector_type(4), aligned(4)));
  typedef double l2_t __attribute__((ext_vector_type(2)));

  __shared__ __attribute__((aligned(16))) double Tr[KW][2][16 * LDT];  // tiles to transpose
  // the waves' first rows, but for their share from the row before; [KW]: what the item's
  // first row gets from there
  __shared__ double Fw[KW + 1][TT][4][64];
  __shared__ double Fa[MN ? KW + 1 : 1][MN ? NB : 1];  // and their row sums of |M|
  __shared__ double red[KW][kParts];

  const ResItem it = items[blockIdx.x];
  const ResSys& S = systems[it.sys];
  const int N = S.N, b0 = it.b0, b1 = it.b1;
  const int w = wave_id(), l = lane_id(), lr = l & 15, lk = l >> 4;
  const long long ND = (long long)NB * nrhs;
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
  // byte offset of a lane behind a uniform base, hidden where it is used (kept over the
  // loop as 64-bit addresses the offsets of all loads would spill)
  auto at = [](auto base, unsigned off) {
    asm volatile("" : "+v"(off));
    return (decltype(base))((const BSS_GLOBAL char*)base + off);
  };

  // -x of block j as A operand: lane (right-hand side lr, row 16 t + 4 lk + q); the
  // right-hand sides that are not there and the blocks outside the system are zero
  struct xraw_t {
    d2_t o[TT][2];
    f4u_t d[TT];
  };
  const int xl = (lr < nrhs ? lr : 0) * NB + 4 * lk;
  auto load_x = [&](xraw_t& v, int j) {
    const long long e = (j < 0 ? 0 : j >= N ? N - 1 : j) * ND;
#pragma unroll
    for (int t = 0; t < TT; ++t) {
      v.d[t] = *(const BSS_GLOBAL f4u_t*)at(dxs + e + 16 * t, 4 * xl);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if constexpr (X0) v.o[t][h] = d2_t{0.0, 0.0};
        else v.o[t][h] = *(const BSS_GLOBAL d2_t*)at(xo + e + 16 * t + 2 * h, 8 * xl);
      }
    }
  };
  auto neg_x = [&](double(&nx)[TT][4], const xraw_t& v, int j) {
    const bool in = j >= 0 && j < N && lr < nrhs;
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const double x = v.o[t][q >> 1][q & 1] + (double)v.d[t][q];
        nx[t][q] = in ? -x : 0.0;
      }
  };
  // d of block j: lane (right-hand side lk + 4 v, row 16 t + lr)
  auto load_d = [&](acc_t(&c)[TT], int j) {
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int k = lk + 4 * v;
        c[t][v] = *at(ds + j * ND + 16 * t, 8 * ((k < nrhs ? k : 0) * NB + lr));
      }
  };
  double rmax[4] = {0, 0, 0, 0}, dmax[4] = {0, 0, 0, 0}, xmax = 0.0, mmax = 0.0;
  auto take_d = [&](acc_t(&c)[TT], bool use) {
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        c[t][v] = use && lk + 4 * v < nrhs ? c[t][v] : 0.0;
        dmax[v] = nmax(dmax[v], fabs(c[t][v]));
      }
  };

  double ring[RING][4];
  const int ml = 4 * lk * NB + lr;  // lane (row lr, column 4 lk + q)
  auto load_tile = [&](double(&u)[4], const BSS_GLOBAL double* blk, int a, int b) {
    const auto g = at(blk + 16 * b * NB + 16 * a, 8 * ml);
#pragma unroll
    for (int q = 0; q < 4; ++q) u[q] = g[q * NB];
  };
  // the tile with rows and columns exchanged: lane (column lr, row 4 lk + q)
  auto transpose = [&](double(&t)[4], const double(&u)[4], double* buf) {
#pragma unroll
    for (int q = 0; q < 4; ++q) buf[(4 * lk + q) * LDT + lr] = u[q];
    fence();
    const l2_t a = *(const l2_t*)(buf + lr * LDT + 4 * lk);
    const l2_t b = *(const l2_t*)(buf + lr * LDT + 4 * lk + 2);
    fence();
    t[0] = a[0];
    t[1] = a[1];
    t[2] = b[0];
    t[3] = b[1];
  };

  double nx[TT][4], np[TT][4];  // -x_i, -x_{i+1}
  acc_t cy[TT], cn[TT];         // row i, row i + 1
  double sy[MN ? TT : 1], sn[MN ? TT : 1];  // row sums of |M| (this lane's share of the columns)

  const int per = (b1 - b0 + KW - 1) / KW;
  const int w0 = b0 + w * per, w1 = min(w0 + per, b1);

  // what row b0 - 1 gives to row b0
  if (w == KW - 1) {
#pragma unroll
    for (int t = 0; t < TT; ++t) {
      cn[t] = Mfma<double>::zero();
      if constexpr (MN) sn[t] = 0.0;
    }
    if (b0 > 0) {
      {
        xraw_t xr;
        load_x(xr, b0 - 1);
        neg_x(nx, xr, b0 - 1);
      }
      // lane (column lr, row 4 lk + q), read as such
#pragma unroll
      for (int b = 0; b < TT; ++b)
#pragma unroll
        for (int a = 0; a < TT; ++a) {
          const auto g = at(Bs + (b0 - 1) * NN + 16 * b * NB + 16 * a, 8 * (lr * NB + 4 * lk));
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const double u = g[q];
            cn[b] = Mfma<double>::mma(nx[a][q], u, cn[b]);
            if constexpr (MN) sn[b] += fabs(u);
          }
        }
    }
#pragma unroll
    for (int t = 0; t < TT; ++t) {
#pragma unroll
      for (int v = 0; v < 4; ++v) Fw[KW][t][v][l] = cn[t][v];
      if constexpr (MN) {
        const double s = row4_sum(sn[t]);
        if (lk == 0) Fa[KW][16 * t + lr] = s;
      }
    }
  }

  auto store_r = [&](long long blk, const acc_t(&c)[TT]) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int k = lk + 4 * v;
      if (k < nrhs) {
#pragma unroll
        for (int t = 0; t < TT; ++t) {
          *at(ro + blk * ND + 16 * t, 4 * (k * NB + lr)) = (float)c[t][v];
          rmax[v] = nmax(rmax[v], fabs(c[t][v]));
        }
      }
    }
  };
  if (w0 < w1) {
    {
      xraw_t xr;
      load_x(xr, w0);
      load_d(cy, w0);
#pragma unroll
      for (int s = 0; s + 1 < RING; ++s)
        if (s < RT::T)
          load_tile(ring[s], RT::is_a(s) ? As + w0 * NN : (w0 + 1 < N ? Bs : As) + w0 * NN,
                    RT::row(s), RT::col(s));
      neg_x(nx, xr, w0);
      // the first row's d comes with the share of the wave before, the item's first row's
      // with this one
      take_d(cy, w == 0);
    }
    if constexpr (MN) {
#pragma unroll
      for (int t = 0; t < TT; ++t) sy[t] = 0.0;
    }
#pragma unroll 1
    for (int i = w0; i < w1; ++i) {
      const bool next = i + 1 < N;
      // the system's last row has no coupling: it reads its A in its place, and drops it
      const auto Ab = As + i * NN, Bb = next ? Bs + i * NN : Ab;
      const int i1 = i + 1 < w1 ? i + 1 : i;  // whose first tiles are loaded last
      const auto An = As + i1 * NN, Bn = i1 + 1 < N ? Bs + i1 * NN : An;
      xraw_t xr;
      load_x(xr, i + 1);
      load_d(cn, i + 1 < b1 ? i + 1 : i);
      if constexpr (MN) {
#pragma unroll
        for (int t = 0; t < TT; ++t) sn[t] = 0.0;
      }
      // x_new of this block
      if (lr < nrhs) {
#pragma unroll
        for (int t = 0; t < TT; ++t)
#pragma unroll
          for (int h = 0; h < 2; ++h)
            *(BSS_GLOBAL d2_t*)at(xn + i * ND + 16 * t + 2 * h, 8 * xl) =
                d2_t{-nx[t][2 * h], -nx[t][2 * h + 1]};
      }
#pragma unroll
      for (int t = 0; t < TT; ++t)
#pragma unroll
        for (int q = 0; q < 4; ++q) xmax = nmax(xmax, fabs(nx[t][q]));

      auto step = [&](auto sc) {
        constexpr int s = decltype(sc)::value;
        constexpr int f = s + RING - 1, fs = f % RT::STEPS;  // the tile to load now
        if constexpr (fs < RT::T) {
          constexpr bool nr = f >= RT::STEPS;
          load_tile(ring[f % RING], RT::is_a(fs) ? (nr ? An : Ab) : (nr ? Bn : Bb), RT::row(fs),
                    RT::col(fs));
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (s == RT::NA) {
          neg_x(np, xr, i + 1);
          take_d(cn, i + 1 < b1);
        }
        if constexpr (s < RT::T) {
          constexpr int a = RT::row(s), b = RT::col(s);
          double(&u)[4] = ring[s % RING];
          // row sums are kept up to date: left to later, they would keep the tiles
          auto settle = [](double& x, double& y) {
            if constexpr (MN) asm volatile("" : "+v"(x), "+v"(y));
          };
          double t[4];
          if constexpr (RT::is_a(s)) {
            transpose(t, u, Tr[w][s & 1]);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              const double ud = a < b || lr <= 4 * lk + q ? u[q] : 0.0;
              const double td = a < b || 4 * lk + q < lr ? t[q] : 0.0;
              cy[a] = Mfma<double>::mma(nx[b][q], ud, cy[a]);
              cy[b] = Mfma<double>::mma(nx[a][q], td, cy[b]);
              if constexpr (MN) {
                sy[a] += fabs(ud);
                sy[b] += fabs(td);
              }
            }
            if constexpr (MN) settle(sy[a], sy[b]);
          } else {
#pragma unroll
            for (int q = 0; q < 4; ++q) u[q] = next ? u[q] : 0.0;
            transpose(t, u, Tr[w][s & 1]);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              cy[a] = Mfma<double>::mma(np[b][q], u[q], cy[a]);
              cn[b] = Mfma<double>::mma(nx[a][q], t[q], cn[b]);
              if constexpr (MN) {
                sy[a] += fabs(u[q]);
                sn[b] += fabs(t[q]);
              }
            }
            if constexpr (MN) settle(sy[a], sn[b]);
          }
        }
      };
      for_each_step(step, std::make_integer_sequence<int, RT::STEPS>{});

      if (i == w0) {
#pragma unroll
        for (int t = 0; t < TT; ++t) {
#pragma unroll
          for (int v = 0; v < 4; ++v) Fw[w][t][v][l] = cy[t][v];
          if constexpr (MN) {
            const double s = row4_sum(sy[t]);
            if (lk == 0) Fa[w][16 * t + lr] = s;
          }
        }
      } else {
        store_r(i, cy);
        if constexpr (MN) {
#pragma unroll
          for (int t = 0; t < TT; ++t) mmax = nmax(mmax, row4_sum(sy[t]));
        }
      }
#pragma unroll
      for (int t = 0; t < TT; ++t) {
        cy[t] = cn[t];
        if constexpr (MN) sy[t] = sn[t];
#pragma unroll
        for (int q = 0; q < 4; ++q) nx[t][q] = np[t][q];
      }
    }
  }
  __syncthreads();
  // the first row of the next wave is finished by this one, the item's by wave 0
  auto finish = [&](int k, long long blk, acc_t(&c)[TT]) {
#pragma unroll
    for (int t = 0; t < TT; ++t) {
#pragma unroll
      for (int v = 0; v < 4; ++v) c[t][v] += Fw[k][t][v][l];
      if constexpr (MN) mmax = nmax(mmax, row4_sum(sy[t]) + Fa[k][16 * t + lr]);
    }
    store_r(blk, c);
  };
  if (w0 < w1 && w1 < b1) finish(w + 1, w1, cy);
  if (w == 0) {
#pragma unroll
    for (int t = 0; t < TT; ++t) {
#pragma unroll
      for (int v = 0; v < 4; ++v) cy[t][v] = Fw[KW][t][v][l];
      if constexpr (MN) sy[t] = lk == 0 ? Fa[KW][16 * t + lr] : 0.0;
    }
    finish(0, b0, cy);
  }
  // maxima: over the rows (lanes lr) of r and d, over lk of x
#pragma unroll
  for (int o = 1; o < 16; o <<= 1) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      rmax[v] = nmax(rmax[v], __shfl_xor(rmax[v], o));
      dmax[v] = nmax(dmax[v], __shfl_xor(dmax[v], o));
    }
    mmax = nmax(mmax, __shfl_xor(mmax, o));
  }
#pragma unroll
  for (int o = 16; o < 64; o <<= 1) {
    xmax = nmax(xmax, __shfl_xor(xmax, o));
    mmax = nmax(mmax, __shfl_xor(mmax, o));
  }
  if (lr == 0) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      red[w][lk + 4 * v] = rmax[v];
      red[w][32 + lk + 4 * v] = dmax[v];
    }
  }
  if (lk == 0) {
    red[w][16 + lr] = xmax;
    red[w][kMnormSlot + lr] = mmax;
  }
  __syncthreads();
  if (threadIdx.x < kParts) {
    double m = red[0][threadIdx.x];
    for (int k = 1; k < KW; ++k) m = nmax(m, red[k][threadIdx.x]);
    part[(long long)blockIdx.x * kParts + threadIdx.x] = m;
  }
}

}  // namespace bss
