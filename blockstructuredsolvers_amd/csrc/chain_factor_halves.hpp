// chain_factor_halves.hpp -- chain factorisation of FP64 factors at block size n = 128.
//
// Same algorithm and outputs as chain_factor_strip_kernel: wave w holds the column strips w
// of B -> C and Z -> W in registers, the block being factored is in LDS as packed upper
// tiles.  One n x n FP64 block is 128 KB here, so the strips that the products exchange
// through LDS go there in halves of four (64 KB beside the triangle's 72 KB, one workgroup
// a CU): first W (S_L += W^T W), then C (Z' = C^T W and A_{i+1} -= C^T C).  A product of
// two strips of different halves takes one from LDS and the other from its wave's
// registers.  The tiles of E that the potrf needs share the exchange area, so nothing of a
// block is left for the next block's windows.
//
// What bounds it: the matrix cores for the solve and the Schur products (two waves share a
// SIMD's), and the eight diagonal tiles in turn between them.  Measured on MI355X, against
// a kernel that kept only the triangle in LDS and staged every product's operands through
// LDS in 16-row slices: 1024 chains of 15 blocks 7.20 -> 5.62 ms, 64 chains (less than
// one a CU) 1.78 -> 1.30 ms.  The three strips take 192 of a lane's 256 registers, and 87
// values (188 bytes a lane) go to scratch all the same; the fences and the sums in memory below
// keep it from more.
#pragma once

#include "chain_factor_strip.hpp"

namespace bss {

template <typename T, int NB>
__global__ void __launch_bounds__(4 * NB) __attribute__((amdgpu_waves_per_eu(2)))
    chain_factor_halves_kernel(FactorLevelArgs p) {
  constexpr int TT = NB / 16, NW = TT, H = TT / 2;
  constexpr long long NN = (long long)NB * NB;
  constexpr int NS = TT * (TT + 1) / 2, NE = TT * (TT - 1) / 2;
  constexpr int HS = H * (H + 1) / 2;           // upper tiles within a half
  constexpr int HQ = (HS + NW - 1) / NW;        // ... per wave
  typedef Img<T> I;
  typedef typename I::tile_t tile_t;
  typedef typename I::vec_t vec_t;
  constexpr int TS = I::SIZE;
  static_assert(NE <= H * TT, "E shares the exchange area");

  __shared__ __attribute__((aligned(16))) T As[NS * TS];      // A, then Uinv (upper tiles)
  __shared__ __attribute__((aligned(16))) T Rs[H * TT * TS];  // E, then half of W or C
  __shared__ __attribute__((aligned(16))) T Es[2 * TS];
  __shared__ __attribute__((aligned(16))) T Is[TS];
  __shared__ int fail;
  auto up = [&](int r, int c) -> T* { return As + (c * (c + 1) / 2 + r) * TS; };
  auto rt = [&](int t, int c) -> T* { return Rs + ((c & (H - 1)) * TT + t) * TS; };

  const ChainRec cd = p.chains[blockIdx.x];
  const int start = cd.start, len = cd.len, sepL = cd.sepL, sepR = cd.sepR;
  if (len <= 0) return;
  const LevelSys S = p.sys[cd.slot];
  const int sys = S.sys;
  const bool hasL = sepL >= 0, hasR = sepR >= 0;
  const auto A = gptr((const T*)S.A);
  const auto B = gptr((const T*)S.B);
  const auto U = gptr((T*)S.U);
  const auto C = gptr((T*)S.C);
  const auto W = gptr((T*)S.W);
  const int w = wave_id();
  const int l = lane_id(), lr = l & 15, lk = l >> 4;
  const int so = I::own_slot(), sa = I::a_slot();
  const TileInverse<T, NB, true> inv{As, Rs, Es, Is, &fail, w, so, sa};
  const int lcol = lr * NB + I::row(lk, 0);  // this lane's elements of a tile in HBM

  // keeps the scheduler from loading more than two steps' operands ahead (they would spill)
  auto fence = [](int t) {
    if (t % 2 == 1) __builtin_amdgcn_sched_barrier(0);
  };
  auto get = [&](const BSS_GLOBAL T* g) -> tile_t {
    tile_t t;
#pragma unroll
    for (int h = 0; h < I::PLANES; ++h) {
      const vec_t x = *gat<const vec_t>(g + 8 * h, lcol);
#pragma unroll
      for (int q = 0; q < I::VEC; ++q) t[I::VEC * h + q] = x[q];
    }
    return t;
  };
  auto put = [&](BSS_GLOBAL T* g, const tile_t& t) {
#pragma unroll
    for (int h = 0; h < I::PLANES; ++h) {
      vec_t x;
#pragma unroll
      for (int q = 0; q < I::VEC; ++q) x[q] = t[I::VEC * h + q];
      *gat<vec_t>(g + 8 * h, lcol) = x;
    }
  };
  // n-th upper tile (a, b) of this wave among those with both strips in the second half
  auto second = [&](int n, int& a, int& b) -> bool {
    const int q = w + NW * n;
    b = 0;
#pragma unroll
    for (int c = 1; c < H; ++c) b += q >= c * (c + 1) / 2 ? 1 : 0;
    a = H + q - b * (b + 1) / 2;
    b += H;
    return q < HS;
  };

  // S_L tiles of this wave: n < H is (n, w), from the first half (n <= w); n >= H is
  // second(n - H).  They are summed up in the S_L slot, in lane order (coalesced, and in L2
  // between blocks): in registers they would spill.
  const auto sl = gptr((T*)S.SL) + (long long)(hasL ? sepL : 0) * NN;
  auto sum_get = [&](int n) -> tile_t {
    tile_t t;
#pragma unroll
    for (int h = 0; h < I::PLANES; ++h) {
      const vec_t x = *gat<const vec_t>(sl + ((w * (H + HQ) + n) * I::PLANES + h) * 64 * I::VEC,
                                        I::VEC * l);
#pragma unroll
      for (int q = 0; q < I::VEC; ++q) t[I::VEC * h + q] = x[q];
    }
    return t;
  };
  auto sum_put = [&](int n, const tile_t& t) {
#pragma unroll
    for (int h = 0; h < I::PLANES; ++h) {
      vec_t x;
#pragma unroll
      for (int q = 0; q < I::VEC; ++q) x[q] = t[I::VEC * h + q];
      *gat<vec_t>(sl + ((w * (H + HQ) + n) * I::PLANES + h) * 64 * I::VEC, I::VEC * l) = x;
    }
  };
  static_assert(NW * (H + HQ) <= TT * TT, "the sums fit the S_L slot");
  // strip w of (-1)^i Z_i, as in chain_factor_strip_kernel
  tile_t Zn[TT];
  if (hasL) {  // Z_1 = B_L^T
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        Zn[t][v] = *gat<const T>(B + (long long)(start - 1) * NN + 16 * t * NB + 16 * w,
                                 I::row(lk, v) * NB + lr);
  } else {
#pragma unroll
    for (int t = 0; t < TT; ++t) Zn[t] = Mfma<T>::zero();
  }
  for (int q = w; q < NS; q += NW) {
    int a = q, b = 0;
    while (a > b) a -= ++b;
    I::store(up(a, b), so, get(A + (long long)start * NN + 16 * b * NB + 16 * a));
  }
  for (int e = threadIdx.x; e < 256; e += 4 * NB)
    Is[I::off(e & 15, e >> 4)] = (e & 15) == (e >> 4) ? T(1) : T(0);
  if (threadIdx.x == 0) fail = 0;
  int fail_i = len;  // first failed block of the chain (thread 0)
  T sg = T(1);       // (-1)^i
  __syncthreads();

  for (int i = 0; i < len; ++i) {
    const long long blk = start + i;
    const bool last = (i == len - 1);
    const bool hasC = !last || hasR;

    inv.windows(U + blk * NN, [](int) {});
    tile_t Cs[TT];
    if (hasC) {
#pragma unroll
      for (int t = 0; t < TT; ++t) Cs[t] = get(B + blk * NN + 16 * w * NB + 16 * t);
    }
    inv.last_window(U + blk * NN);
    __syncthreads();
    if (threadIdx.x == 0 && fail) {
      fail_i = min(fail_i, i);
      fail = 0;
    }

    // [C | W] strips, in place from the last row tile up
    tile_t Ws[TT];
#pragma unroll
    for (int t = 0; t < TT; ++t) Ws[t] = Zn[t];
    auto trsm = [&](auto with_w) {
#pragma unroll
      for (int r = TT - 1; r >= 0; --r) {
        tile_t c = Mfma<T>::zero(), z = Mfma<T>::zero();
#pragma unroll
        for (int t = 0; t <= r; ++t) {
          const tile_t x = I::load(up(t, r), sa);
          mma16<T>(c, x, Cs[t]);
          if constexpr (decltype(with_w)::value) mma16<T>(z, x, Ws[t]);
          fence(t);
        }
        Cs[r] = c;
        if constexpr (decltype(with_w)::value) Ws[r] = z;
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    if (hasL)
      trsm(yes_t());
    else
      trsm(no_t());

    // half h of the strips to LDS and, times f, to HBM (out: null = not there).  The first
    // barrier: the exchange area is free (E, the other strips' reads); the second: filled.
    auto exchange = [&](int h, const tile_t (&X)[TT], BSS_GLOBAL T* out, T f) {
      __syncthreads();
      if ((w >= H) == (h == 1)) {
#pragma unroll
        for (int t = 0; t < TT; ++t) I::store(rt(t, w), so, X[t]);
      }
      __syncthreads();
      if ((w >= H) == (h == 1)) {
        if (f > T(0))
          put_tiles<T, NB, TT>(out + 16 * w * NB, rt(0, w));
        else
          put_tiles<T, NB, TT, true>(out + 16 * w * NB, rt(0, w));
      }
    };
    if (hasL) {  // S_L += W^T W
      exchange(0, Ws, W + blk * NN, sg);
#pragma unroll
      for (int a = 0; a < H; ++a) {
        if (a <= w) {
          const tile_t s = sum_get(a);  // (undefined before the first block's sum)
          tile_t c = Mfma<T>::zero();
#pragma unroll
          for (int t = 0; t < TT; ++t) {
            mma16<T>(c, I::load(rt(t, a), sa), Ws[t]);
            fence(t);
          }
          sum_put(a, i > 0 ? s + c : c);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      exchange(1, Ws, W + blk * NN, sg);
#pragma unroll
      for (int n = 0; n < HQ; ++n) {
        int a, b;
        if (second(n, a, b)) {
          const tile_t s = sum_get(H + n);
          tile_t c = Mfma<T>::zero();
#pragma unroll
          for (int t = 0; t < TT; ++t) {
            mma16<T>(c, I::load(rt(t, a), sa), I::load(rt(t, b), so));
            fence(t);
          }
          sum_put(H + n, i > 0 ? s + c : c);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (hasC) {
      // Z'(a, w) = C_a^T W_w (its sign left out);  C_a^T C_b into A_{i+1}(a, b), or to S_R
      // after the last block;  B' = -W_last^T C_last is -Z' transposed
      const auto An = A + (last ? blk : blk + 1) * NN;
      const auto sr = gptr((T*)S.SR) + (long long)(hasR ? sepR : 0) * NN;
      auto diag_out = [&](int a, int b, const tile_t& x, const tile_t& c) {
        if (!last)
          I::store(up(a, b), so, x - c);
        else
          put(sr + 16 * b * NB + 16 * a, c);
      };
      auto z_out = [&](int a, const tile_t& z) {
        Zn[a] = z;
        if (last) {
          const auto g = gptr((T*)S.Bn) + (long long)sepL * NN + 16 * a * NB + 16 * w;
#pragma unroll
          for (int v = 0; v < 4; ++v) *gat<T>(g, I::row(lk, v) * NB + lr) = -sg * z[v];
        }
      };
      exchange(0, Cs, C + blk * NN, T(1));
      auto first_half = [&](auto with_z) {
        constexpr bool Z = decltype(with_z)::value;
#pragma unroll
        for (int a = 0; a < H; ++a) {
          tile_t z = Mfma<T>::zero(), c = Mfma<T>::zero();
          if (a <= w) {
            const tile_t x = get(An + 16 * w * NB + 16 * a);
#pragma unroll
            for (int t = 0; t < TT; ++t) {
              const tile_t y = I::load(rt(t, a), sa);
              mma16<T>(c, y, Cs[t]);
              if constexpr (Z) mma16<T>(z, y, Ws[t]);
              fence(t);
            }
            diag_out(a, w, x, c);
          } else if constexpr (Z) {
#pragma unroll
            for (int t = 0; t < TT; ++t) {
              mma16<T>(z, I::load(rt(t, a), sa), Ws[t]);
              fence(t);
            }
          }
          if constexpr (Z) z_out(a, z);
          __builtin_amdgcn_sched_barrier(0);
        }
      };
      if (hasL)
        first_half(yes_t());
      else
        first_half(no_t());
      exchange(1, Cs, C + blk * NN, T(1));
#pragma unroll
      for (int n = 0; n < HQ; ++n) {
        int a, b;
        if (second(n, a, b)) {
          const tile_t x = get(An + 16 * b * NB + 16 * a);
          tile_t c = Mfma<T>::zero();
#pragma unroll
          for (int t = 0; t < TT; ++t) {
            mma16<T>(c, I::load(rt(t, a), sa), I::load(rt(t, b), so));
            fence(t);
          }
          diag_out(a, b, x, c);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      if (hasL) {
#pragma unroll
        for (int a = H; a < TT; ++a) {
          tile_t z = Mfma<T>::zero();
#pragma unroll
          for (int t = 0; t < TT; ++t) {
            mma16<T>(z, I::load(rt(t, a), sa), Ws[t]);
            fence(t);
          }
          z_out(a, z);
          __builtin_amdgcn_sched_barrier(0);
        }
      } else {
        forget(Zn);
      }
    }
    // (window -1 of the next block reads tile (0, 0), written by this wave or ahead of the
    // last exchange, and its barrier comes before E is written)
    sg = -sg;
  }
  if (hasL) {  // the sums into column-major order, over the same memory
    tile_t Sl[H + HQ];
#pragma unroll
    for (int n = 0; n < H + HQ; ++n) Sl[n] = sum_get(n);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
#pragma unroll
    for (int n = 0; n < H; ++n)
      if (n <= w) put(sl + 16 * w * NB + 16 * n, Sl[n]);
#pragma unroll
    for (int n = 0; n < HQ; ++n) {
      int a, b;
      if (second(n, a, b)) put(sl + 16 * b * NB + 16 * a, Sl[H + n]);
    }
  }
  // original indices increase along a chain: the first local failure is the smallest
  if (threadIdx.x == 0 && fail_i < len) {
    const int blk = start + fail_i;
    atomicMin(p.info + sys, (S.orig ? S.orig[blk] : blk) + 1);
  }
}

}  // namespace bss
