// chain_factor_strip.hpp -- fused per-chain factorisation with column strips in registers.
//
// Same algorithm and outputs as described in chain_factor.hpp; wave w of the chain's
// n/16 waves owns the 16-column strips w of B -> C and of Z -> W and holds them in
// registers from their load (or their product) to their store:
//   trsm    [C | W] strip = Uinv^T [B | Z] strip      Uinv tiles from LDS, strips in place
//   Schur   Z' strip = C^T W strip                    C tiles from LDS, own W strip
//           A_{i+1} column strip n/16-1-w -= C^T C    C tiles from LDS
//           S_L column strip w += W^T W strip         W tiles from LDS, own W strip
// Only the block being factored and one n x n block of C (later W) are in LDS, so two
// FP64 chains of n = 64 share a CU (72 KB each; a kernel with A, Uinv, C and W whole in
// LDS took 135 KB and held one) and the products of one run beside the serial 16x16
// diagonal steps of another.  Within a chain too: what no later step of the potrf waits for
// (Z', S_L, the rows off the next diagonal tile) runs on the waves that do not hold the
// current diagonal tile.
//
// What bounds it: per block the 4 to 8 diagonal tiles in turn (3.2K cycles each in FP64,
// 2.5K in FP32, more beside other waves' MFMAs) and the products: at n = 64 in FP64 the matrix
// cores are busy in 62% of the cycles and do 51% of their peak rate.  Measured on MI355X, level-0 factorisation of 32 systems, N = 8192,
// n = 64, against the whole-block kernel before it: FP64 18.16 -> 12.2 ms, FP32 factors
// of FP64 input with the fused forward sweep 9.13 -> 7.08 ms; 24 systems of n = 32, FP64:
// 0.53 -> 0.29 ms; n = 48, FP32, 98 blocks in one chain: 0.90 -> 0.61 ms; n = 96, FP32
// factors, 8 systems of 2048 blocks: 1.74 -> 1.61 ms.
//
// Every product is X^T Y over 16x16 tiles.  A register tile holds element (row(lk, v), lr)
// in register v of lane (lr, lk) = (l % 16, l / 16) ("P layout", Img below).  That is the B
// operand of X^T Y as it stands (k slot lk of step v is row(lk, v)), and a tile dumped to
// LDS lane by lane reads back as the A operand: lane (lr, lk) supplies X[row(lk, v)][lr].
// The FP64 MFMA returns the product's row lk + 4 v in register v (the FP32 one 4 lk + v),
// so the FP64 A operand is read with its columns permuted (a_col): the product then comes
// out in P layout too.
#pragma once

#include "chain_factor.hpp"

namespace bss {

// One 16x16 tile in LDS (256 elements) as the register image of a wave in P layout: lane
// (lr, lk) holds column lr, rows row(lk, v) in register v.  16-byte vectors of two (FP64,
// in two planes) or four (FP32) rows, vector (lr, lk) of a plane in slot
// 16 lk + (lr + lk) % 16: a whole wave reads or writes a tile, its A operand, and (for the
// HBM stores) the vectors of a column by consecutive lanes without bank conflicts.
template <typename T>
struct Img {
  typedef typename Mfma<T>::acc_t tile_t;
  static constexpr int SIZE = 256;
  static constexpr int VEC = 16 / sizeof(T);  // rows per vector
  typedef T vec_t __attribute__((ext_vector_type(VEC)));
  static constexpr int PLANES = 4 / VEC;
  __device__ static constexpr int row(int lk, int v) {
    return sizeof(T) == 4 ? 4 * lk + v : 8 * (v >> 1) + 2 * lk + (v & 1);
  }
  __device__ static inline int slot(int lr, int lk) { return 16 * lk + ((lr + lk) & 15); }
  // offset of element (r, c)
  __device__ static inline int off(int r, int c) {
    if constexpr (sizeof(T) == 4)
      return 4 * slot(c, r >> 2) + (r & 3);
    else
      return 128 * (r >> 3) + 2 * slot(c, (r & 7) >> 1) + (r & 1);
  }
  // this lane's slots: its own and its A operand's
  __device__ static inline int own_slot() { return slot(lane_id() & 15, lane_id() >> 4); }
  // the column whose vectors are this lane's A operand
  __device__ static inline int a_col() {
    const int i = lane_id() & 15;
    return sizeof(T) == 4 ? i : (i & 8) + 2 * (i & 3) + ((i >> 2) & 1);
  }
  __device__ static inline int a_slot() { return slot(a_col(), lane_id() >> 4); }
  __device__ static inline tile_t load(const T* p, int slot) {
    if constexpr (sizeof(T) == 4) {
      return *(const vec_t*)(p + 4 * slot);
    } else {
      const vec_t a = *(const vec_t*)(p + 2 * slot), b = *(const vec_t*)(p + 128 + 2 * slot);
      return tile_t{a[0], a[1], b[0], b[1]};
    }
  }
  __device__ static inline void store(T* p, int slot, const tile_t& t) {
    if constexpr (sizeof(T) == 4) {
      *(vec_t*)(p + 4 * slot) = t;
    } else {
      *(vec_t*)(p + 2 * slot) = vec_t{t[0], t[1]};
      *(vec_t*)(p + 128 + 2 * slot) = vec_t{t[2], t[3]};
    }
  }
};

// The tiles get no defined value but count as written: ends their live range where every
// later use is behind a write that the compiler cannot see to be always taken.
template <typename V, int N>
__device__ __attribute__((always_inline)) inline void forget(V (&t)[N]) {
#pragma unroll
  for (int k = 0; k < N; ++k) asm volatile("" : "=v"(t[k]));
}

// acc += X^T Y over one 16-deep step, X as A operand, Y in P layout
template <typename T>
__device__ inline void mma16(typename Mfma<T>::acc_t& acc, const typename Mfma<T>::acc_t& a,
                             const typename Mfma<T>::acc_t& b) {
#pragma unroll
  for (int q = 0; q < 4; ++q) acc = Mfma<T>::mma(a[q], b[q], acc);
}

// the sweeps' dot product (XOps::dot of chain_solve.hpp) over one 16-deep slice
template <typename T>
__device__ inline void dot16(T& t0, T& t1, const typename Mfma<T>::acc_t& x, const T* y) {
  t0 = fma(x[0], y[0], t0);
  t1 = fma(x[1], y[1], t1);
  t0 = fma(x[2], y[2], t0);
  t1 = fma(x[3], y[3], t1);
}

struct yes_t {
  static constexpr bool value = true;
};
struct no_t {
  static constexpr bool value = false;
};

// 16 bytes of global memory
template <typename T>
struct Vec16 {
  static constexpr int N = 16 / sizeof(T);
  typedef T type __attribute__((ext_vector_type(N)));
};

// element `off` (per lane, non-negative) behind a wave-uniform base.  The byte offset is
// hidden from the optimiser where it is used, so that it stays a 32-bit register beside a
// scalar base: widened ahead of the block loop, the 64-bit lane addresses would spill.
template <typename V, typename P>
__device__ __attribute__((always_inline)) inline BSS_GLOBAL V* gat(P base, int off) {
  return (BSS_GLOBAL V*)((BSS_GLOBAL char*)base + (unsigned)opaque_v(off * (int)sizeof(*base)));
}

// d += (lane R of each 16-lane row of m) * f.  One instruction where a DPP move and an FMA
// take two; the compiler does not fold the 64-bit move.  The caller keeps two wait states
// between the write of m and the first use.
template <int R>
__device__ __attribute__((always_inline)) inline void fmac_lane(double& d, double m, double f) {
  asm volatile("v_fmac_f64_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
               : "+v"(d)
               : "v"(m), "v"(f), "n"(R));
}
template <int R>
__device__ __attribute__((always_inline)) inline void fmac_lane(float& d, float m, float f) {
  asm volatile("v_fmac_f32_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
               : "+v"(d)
               : "v"(m), "v"(f), "n"(R));
}
template <int R0, int R1, typename T>
__device__ __attribute__((always_inline)) inline void fmac_rows(T (&v)[16], T m, T f) {
  if constexpr (R0 < R1 && R0 < 16) {
    fmac_lane<R0>(v[R0], m, f);
    fmac_rows<R0 + 1, R1>(v, m, f);
  }
}
// rows 0, 0, 2, 2 of x in the four 16-lane rows
__device__ inline unsigned even_rows(unsigned x) {
  return __builtin_amdgcn_permlane16_swap(x, x, false, false)[0];
}
__device__ inline float even_rows(float x) {
  return __uint_as_float(even_rows(__float_as_uint(x)));
}
__device__ inline double even_rows(double x) {
  return __hiloint2double((int)even_rows((unsigned)__double2hiint(x)),
                          (int)even_rows((unsigned)__double2loint(x)));
}
// x with lane L replaced by the wave-uniform v.  By the intrinsic (clang has no builtin for
// it): two wait states have to lie between the lane read that writes v's SGPR and this read of
// it, and the compiler keeps them only where it sees the instruction.
__device__ int llvm_writelane(int v, int lane, int x) __asm("llvm.amdgcn.writelane.i32");
template <int L>
__device__ __attribute__((always_inline)) inline int write_lane(int x, int v) {
  return llvm_writelane(__builtin_amdgcn_readfirstlane(v), L, x);
}
template <int L>
__device__ __attribute__((always_inline)) inline float write_lane(float x, float v) {
  return __int_as_float(write_lane<L>(__float_as_int(x), __float_as_int(v)));
}
template <int L>
__device__ __attribute__((always_inline)) inline double write_lane(double x, double v) {
  return __hiloint2double(write_lane<L>(__double2hiint(x), __double2hiint(v)),
                          write_lane<L>(__double2loint(x), __double2loint(v)));
}

// Elimination steps of the 16x16 tile.  Every lane holds a column v[0..15]: in the even
// 16-lane rows column c = lane % 16 of A, in the odd ones column c of the identity, which
// becomes that of E.  Step J subtracts A[J][r] / A[J][J] times row J from the rows r > J
// of both at once: m (row J of A in every 16-lane row) supplies the multipliers by DPP,
// f = -v[J] / A[J][J] is the lane's own factor.  One FMA per row serves A and E (the same
// steps on separate A and E registers take twice the FMAs, which a wave shares its SIMD's
// issue slots for with the other waves' MFMAs).  Only the upper part of A is read.  The
// scaling by 1 / sqrt of the pivots (gathered in pv) is left to the end.  The next step's
// pivot chain is interleaved with this step's rows by hand: sched_barrier keeps the order.
// WIDE: m and f have 1 / sqrt of the pivot each, for any pivot: 1 / A[J][J] on f alone is
// denormal for a pivot in the top binades (FP32's rcp returns zero above 2^126), and with a
// large E overflows for one in the bottom binades.
template <int J, bool WIDE>
__device__ __attribute__((always_inline)) inline void elim_step(double (&v)[16], double m,
                                                                double f, double& pv) {
  if constexpr (J < 15) {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_nop 1");
    fmac_rows<J + 1, J + 2>(v, m, f);
    __builtin_amdgcn_sched_barrier(0);
    fmac_rows<J + 2, J + 3>(v, m, f);
    __builtin_amdgcn_sched_barrier(0);
    const double p = read_lane(v[J + 1], J + 1);
    double mn = even_rows(v[J + 1]);
    __builtin_amdgcn_sched_barrier(0);
    fmac_rows<J + 3, J + 4>(v, m, f);
    __builtin_amdgcn_sched_barrier(0);
    // about 2^-24; third-order step below
    const double y = WIDE ? __builtin_amdgcn_rsq(p) : __builtin_amdgcn_rcp(p);
    __builtin_amdgcn_sched_barrier(0);
    fmac_rows<J + 4, J + 6>(v, m, f);
    __builtin_amdgcn_sched_barrier(0);
    const double py = WIDE ? p * y : p;
    __builtin_amdgcn_sched_barrier(0);
    fmac_rows<J + 6, J + 7>(v, m, f);
    __builtin_amdgcn_sched_barrier(0);
    const double e = fma(-py, y, 1.0), g = v[J + 1] * y;
    if constexpr (WIDE) mn *= y;
    pv = write_lane<J + 1>(pv, p);
    __builtin_amdgcn_sched_barrier(0);
    fmac_rows<J + 7, J + 8>(v, m, f);
    __builtin_amdgcn_sched_barrier(0);
    const double t = fma(e, e, e);
    __builtin_amdgcn_sched_barrier(0);
    fmac_rows<J + 8, J + 9>(v, m, f);
    __builtin_amdgcn_sched_barrier(0);
    const double fn = fma(-g, t, -g);
    __builtin_amdgcn_sched_barrier(0);
    fmac_rows<J + 9, 16>(v, m, f);
    elim_step<J + 1, WIDE>(v, mn, fn, pv);
  }
}
template <int J, bool WIDE>
__device__ __attribute__((always_inline)) inline void elim_step(float (&v)[16], float m, float f,
                                                                float& pv) {
  if constexpr (J < 15) {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_nop 1");
    fmac_rows<J + 1, J + 2>(v, m, f);
    __builtin_amdgcn_sched_barrier(0);
    fmac_rows<J + 2, J + 3>(v, m, f);
    __builtin_amdgcn_sched_barrier(0);
    const float p = read_lane(v[J + 1], J + 1);
    float mn = even_rows(v[J + 1]);
    __builtin_amdgcn_sched_barrier(0);
    fmac_rows<J + 3, J + 4>(v, m, f);
    __builtin_amdgcn_sched_barrier(0);
    // 1 ulp, as the sweep's other roundings
    const float y = WIDE ? __builtin_amdgcn_rsqf(p) : __builtin_amdgcn_rcpf(p);
    pv = write_lane<J + 1>(pv, p);
    __builtin_amdgcn_sched_barrier(0);
    fmac_rows<J + 4, J + 7>(v, m, f);
    __builtin_amdgcn_sched_barrier(0);
    const float fn = -(v[J + 1] * y);
    if constexpr (WIDE) mn *= y;
    __builtin_amdgcn_sched_barrier(0);
    fmac_rows<J + 7, 16>(v, m, f);
    elim_step<J + 1, WIDE>(v, mn, fn, pv);
  }
}
template <bool WIDE>
__device__ __attribute__((always_inline)) inline void eliminate(double (&v)[16], double& pv) {
  const double p = read_lane(v[0], 0);
  const double y = WIDE ? __builtin_amdgcn_rsq(p) : __builtin_amdgcn_rcp(p);
  const double e = fma(-(WIDE ? p * y : p), y, 1.0), g = v[0] * y;
  pv = write_lane<0>(1.0, p);
  elim_step<0, WIDE>(v, WIDE ? even_rows(v[0]) * y : even_rows(v[0]), fma(-g, fma(e, e, e), -g),
                     pv);
}
template <bool WIDE>
__device__ __attribute__((always_inline)) inline void eliminate(float (&v)[16], float& pv) {
  const float p = read_lane(v[0], 0);
  const float y = WIDE ? __builtin_amdgcn_rsqf(p) : __builtin_amdgcn_rcpf(p);
  pv = write_lane<0>(1.0f, p);
  elim_step<0, WIDE>(v, WIDE ? even_rows(v[0]) * y : even_rows(v[0]), -(v[0] * y), pv);
}
// whether x is in [2^-1000, 2^1000) (FP32: [2^-100, 2^100))
__device__ inline bool mid_range(double x) {
  return (unsigned)__double2hiint(x) - (23u << 20) < (2000u << 20);
}
__device__ inline bool mid_range(float x) {
  return __float_as_uint(x) - (27u << 23) < (200u << 23);
}
template <int R, typename T>
__device__ __attribute__((always_inline)) inline void scale_rows(T (&v)[16], T s) {
  if constexpr (R < 16) {
    v[R] *= row_bcast<R>(s);
    scale_rows<R + 1>(v, s);
  }
}

// Cholesky + inverse of the symmetric 16x16 tile with image `at` (upper part): the image of
// Uinv = U^-1 (strict lower part exact zeros) to `ut` (may be `at`), the image of E = Uinv^T
// to `et`; `eye` is the image of the identity.  Returns false if a pivot was not positive.
// One unsigned comparison of the exponents finds the pivots that are not positive and those
// whose reciprocal may leave the exponent range (the first of either is itself right); for the
// latter the tile is done again, WIDE.  WIDE in every tile takes 1% off a small FP64 system (n
// = 32, 100 blocks: 104.5 -> 105.7 us; this 105.0), and loses 2% of the accuracy of FP64
// tiles.  ALWAYS_WIDE: the same, for a kernel in which the second try's registers spill (FP64
// at n = 128, 16 right-hand sides: 5.24 -> 5.24 ms, with the second try 5.30 to 5.51).
template <typename T, bool ALWAYS_WIDE>
__device__ __attribute__((always_inline)) inline bool diag_img(const T* at, T* ut, T* et,
                                                               const T* eye) {
  typedef Img<T> I;
  const int c = opaque_v(lane_id() & 15);
  T v[16], pv;
  auto load = [&](int c) {
    const T* src = (lane_id() >> 4) & 1 ? eye : at;
#pragma unroll
    for (int g = 0; g < 16 / I::VEC; ++g) {
      const auto t = *(const typename I::vec_t*)(src + I::off(I::VEC * g, c));
#pragma unroll
      for (int q = 0; q < I::VEC; ++q) v[I::VEC * g + q] = t[q];
    }
  };
  load(c);
  eliminate<ALWAYS_WIDE>(v, pv);
  T s = rsqrt_nr(pv);
  bool ok = true;
  if (__builtin_amdgcn_ballot_w64(!mid_range(pv)) != 0) {
    if constexpr (!ALWAYS_WIDE) {
      if (__builtin_amdgcn_ballot_w64(pv > T(0) && !mid_range(pv)) != 0) {
        load(opaque_v(lane_id() & 15));
        eliminate<true>(v, pv);
        s = rsqrt_nr(pv);
      }
    }
    ok = __builtin_amdgcn_ballot_w64(!(pv > T(0))) == 0;
  }
  __builtin_amdgcn_sched_barrier(0);
  scale_rows<0>(v, even_rows(s));
  if ((lane_id() >> 4) == 1) {  // E[r][c] = Uinv[c][r] in v[r]
#pragma unroll
    for (int r = 0; r < 16; ++r) ut[I::off(c, r)] = v[r];
#pragma unroll
    for (int g = 0; g < 16 / I::VEC; ++g) {
      typename I::vec_t t;
#pragma unroll
      for (int q = 0; q < I::VEC; ++q) t[q] = v[I::VEC * g + q];
      *(typename I::vec_t*)(et + I::off(I::VEC * g, c)) = t;
    }
  }
  return ok;
}

// N tiles, one below the other, from consecutive images in LDS to HBM (column-major, leading
// dimension NB), negated if NEG.  Lane l takes column l / 4, vector l % 4: four lanes write
// 64 contiguous bytes.  A store from the registers' own lane order (column l % 16) takes 64
// cycles instead of 20 (1 KB, one CU).  The lane's addresses are formed once: beside the
// MFMAs of the SIMD's other waves every vector instruction waits for one of them.
template <typename T, int NB, int N, bool NEG = false>
__device__ __attribute__((always_inline)) inline void put_tiles(BSS_GLOBAL T* g, const T* tiles) {
  typedef Img<T> I;
  typedef typename I::vec_t vec_t;
  const int l = opaque_v(lane_id());
  const unsigned off = (unsigned)opaque_v(((l >> 2) * NB + I::VEC * (l & 3)) * (int)sizeof(T));
  const T* src = tiles + I::VEC * I::slot(l >> 2, l & 3);
#pragma unroll
  for (int t = 0; t < N; ++t)
#pragma unroll
    for (int h = 0; h < I::PLANES; ++h) {
      const vec_t x = *(const vec_t*)(src + I::SIZE * t + 128 * h);
      *(BSS_GLOBAL vec_t*)((BSS_GLOBAL char*)(g + 16 * t + 8 * h) + off) = NEG ? -x : x;
    }
}

// potrf and inverse of the n x n block whose upper tiles are in As (packed by columns), by
// the workgroup's n/16 waves; on return they hold Uinv = U^-1, and so does HBM.  Ls: tiles
// E(i, t), t < i, of E = U^-T; Es: diagonal tiles of E, two in turn (the first is written
// while other waves may still read what shares Ls's memory); Is: the identity.
//
// Windows k = -1 .. TT-1, one barrier each (the last one the caller's).  In window
// k < TT-1 wave k+1 updates diagonal tile k+1 with row k and factors it.  The other waves
// use Uinv_kk, published by window k-1: row i > k takes A(i, j) -= U_ki^T U_kj and
// E(i, t) -= U_ki^T E_kt, one row a wave, and the waves left over finish Uinv(t, k).  Every
// wave forms the tiles of row k that it needs itself (U_kj = Uinv_kk^T A_kj), so that row
// k is never rewritten and one barrier per diagonal tile is enough; with a row-scaling
// phase and its barrier the FP64 factorisation at n = 64 took 13.6 ms where it takes 12.2.
// `extra(k)` is the caller's own work in window k.
template <typename T, int NB, bool ALWAYS_WIDE = false>
struct TileInverse {
  typedef Img<T> I;
  typedef typename I::tile_t tile_t;
  static constexpr int TT = NB / 16, TS = I::SIZE;
  T *As, *Ls, *Es;
  const T* Is;
  int* fail;
  int w, so, sa;

  __device__ inline T* up(int r, int c) const { return As + (c * (c + 1) / 2 + r) * TS; }
  __device__ inline T* lo(int i, int t) const { return Ls + (i * (i - 1) / 2 + t) * TS; }
  __device__ inline T* ed(int k) const { return Es + (k & 1) * TS; }

  // Uinv(u, k) = (Uinv_kk^T E(k, u))^T, to LDS and HBM
  __device__ __attribute__((always_inline)) inline void finish(BSS_GLOBAL T* U, int u, int k,
                                                               const tile_t& x) const {
    tile_t e = Mfma<T>::zero();
    mma16<T>(e, x, I::load(lo(k, u), so));
    const auto g = U + 16 * k * NB + 16 * u;
    const int olr = opaque_v(lane_id() & 15), olk = opaque_v(lane_id() >> 4);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      up(u, k)[I::off(olr, I::row(olk, v))] = e[v];
      *gat<T>(g + I::row(0, v) * NB, I::row(olk, 0) * NB + olr) = e[v];
    }
  }
  __device__ __attribute__((always_inline)) inline void put_diag(BSS_GLOBAL T* U, int k) const {
    put_tiles<T, NB, 1>(U + 16 * k * NB + 16 * k, up(k, k));
  }

  template <typename Extra>
  __device__ __attribute__((always_inline)) inline void windows(BSS_GLOBAL T* U, Extra extra) const {
#pragma unroll 1
    for (int k = -1; k < TT - 1; ++k) {
      if (w == k + 1) {
        if (k >= 0) {
          const tile_t x = I::load(up(k, k), sa);
          tile_t ub = Mfma<T>::zero(), acc = I::load(up(w, w), so);
          mma16<T>(ub, x, I::load(up(k, w), so));
          if constexpr (sizeof(T) == 4) {
            mma16<T>(acc, -ub, ub);
          } else {
            tile_t ua = Mfma<T>::zero();
            mma16<T>(ua, x, I::load(up(k, w), sa));
            mma16<T>(acc, -ua, ub);
          }
          I::store(up(w, w), so, acc);
        }
        if (!diag_img<T, ALWAYS_WIDE>(up(w, w), up(w, w), ed(w), Is) && lane_id() == 0) *fail = 1;
      } else if (k >= 0) {
        const tile_t x = I::load(up(k, k), sa);
        const int u = w - (w > k + 1 ? 1 : 0);
        if (u < k) {
          finish(U, u, k, x);
        } else {
          const int r = u + 1;  // row r > k
          tile_t ua = Mfma<T>::zero();
          mma16<T>(ua, x, I::load(up(k, r), sa));
          ua = -ua;
          for (int j = (r == k + 1 ? r + 1 : r); j < TT; ++j) {
            tile_t ub = Mfma<T>::zero(), acc = I::load(up(r, j), so);
            mma16<T>(ub, x, I::load(up(k, j), so));
            mma16<T>(acc, ua, ub);
            I::store(up(r, j), so, acc);
          }
          for (int t = 0; t < k; ++t) {
            tile_t eb = Mfma<T>::zero(), acc = I::load(lo(r, t), so);
            mma16<T>(eb, x, I::load(lo(k, t), so));
            mma16<T>(acc, ua, eb);
            I::store(lo(r, t), so, acc);
          }
          tile_t acc = Mfma<T>::zero();
          mma16<T>(acc, ua, I::load(ed(k), so));
          I::store(lo(r, k), so, acc);
        }
        if (w == k) put_diag(U, k);
      }
      extra(k);
      __syncthreads();
    }
  }
  __device__ __attribute__((always_inline)) inline void last_window(BSS_GLOBAL T* U) const {
    const tile_t x = I::load(up(TT - 1, TT - 1), sa);
    if (w < TT - 1)
      finish(U, w, TT - 1, x);
    else
      put_diag(U, TT - 1);
  }
};

// Waves per SIMD the registers are budgeted for (512 / this), from the workgroups that LDS
// lets share a CU.  Three variants spill: n = 96 FP64 (22 registers, 84 bytes a lane) and FP32
// factors of FP64 input with the forward sweep at n = 96 (17, 40) and n = 48 (6, 28).
template <typename T, int NB>
constexpr int strip_waves_per_eu() {
  if (sizeof(T) == 8) return NB >= 48 ? 2 : 3;
  return NB == 128 ? 2 : NB >= 64 ? 3 : 4;
}

template <typename Tin, typename T, int NB, bool FWD = false>
__global__ void __launch_bounds__(4 * NB)
    __attribute__((amdgpu_waves_per_eu(strip_waves_per_eu<T, NB>())))
    chain_factor_strip_kernel(FactorLevelArgs p) {
  constexpr int TT = NB / 16, NW = TT;
  constexpr long long NN = (long long)NB * NB;
  constexpr int NS = TT * (TT + 1) / 2, NE = TT * (TT - 1) / 2;
  constexpr int SQ = 1 + (NE + NW - 1) / NW;  // upper tiles per wave
  // When the input is loaded: B before the last diagonal tile's barrier and A before the
  // solve, or (LATE, where those registers spill) B in two halves before the solve and A
  // after it
  constexpr bool LATE = TT >= 6;
  // W has tiles of its own in LDS up to n = 48; above that it takes C's place
  constexpr bool OWN_W = TT <= 3;
  typedef Img<T> I;
  typedef typename I::tile_t tile_t;
  // a lane's four elements of a tile in the input: vectors of 16 bytes
  typedef typename Vec16<Tin>::type inv_t;
  constexpr int IV = Vec16<Tin>::N, IP = 4 / IV;
  typedef typename I::vec_t outv_t;
  constexpr int TS = I::SIZE;

  __shared__ __attribute__((aligned(16))) T As[NS * TS];       // A, then Uinv (upper tiles)
  __shared__ __attribute__((aligned(16))) T Rs[TT * TT * TS];  // C, then W
  __shared__ __attribute__((aligned(16))) T Vs[OWN_W ? TT * TT * TS : 1];
  __shared__ __attribute__((aligned(16))) T Ls[NE > 0 ? NE * TS : 1];  // E(i, t), t < i
  __shared__ __attribute__((aligned(16))) T Es[2 * TS];        // diagonal tiles of E, in turn
  __shared__ T Fr[FWD ? NB : 1], Fy[FWD ? NB : 1];
  __shared__ __attribute__((aligned(16))) T Is[TS];            // the identity
  __shared__ int fail;
  auto up = [&](int r, int c) -> T* { return As + (c * (c + 1) / 2 + r) * TS; };
  auto ct = [&](int t, int c) -> T* { return Rs + (c * TT + t) * TS; };
  auto wt = [&](int t, int c) -> T* { return (OWN_W ? Vs : Rs) + (c * TT + t) * TS; };

  const ChainRec cd = p.chains[blockIdx.x];
  const int start = cd.start, len = cd.len, sepL = cd.sepL, sepR = cd.sepR;
  if (len <= 0) return;
  const LevelSys S = p.sys[cd.slot];
  const int sys = S.sys;
  const bool hasL = sepL >= 0, hasR = sepR >= 0;
  const auto A = gptr((const Tin*)S.A);
  const auto B = gptr((const Tin*)S.B);
  const auto U = gptr((T*)S.U);
  const auto C = gptr((T*)S.C);
  const auto W = gptr((T*)S.W);
  const int w = wave_id();
  const int l = lane_id(), lr = l & 15, lk = l >> 4;
  const int so = I::own_slot(), sa = I::a_slot();
  const TileInverse<T, NB> inv{As, Ls, Es, Is, &fail, w, so, sa};
  // this lane's elements of a tile in global memory: its first vector (the second is
  // DIV rows further)
  constexpr int DIV = sizeof(T) == 4 ? IV : 8;
  const int lcol = lr * NB + I::row(lk, 0);

  struct raw_t {
    inv_t p[IP];
  };
  auto load_raw = [&](const BSS_GLOBAL Tin* g) -> raw_t {
    raw_t r;
#pragma unroll
    for (int h = 0; h < IP; ++h) r.p[h] = *gat<const inv_t>(g + DIV * h, lcol);
    return r;
  };
  auto cvt = [](const raw_t& r) -> tile_t {
    tile_t t;
#pragma unroll
    for (int v = 0; v < 4; ++v) t[v] = (T)r.p[v / IV][v % IV];
    return t;
  };
  // This wave's upper tiles (a, b) of a symmetric block: n = 0 is its diagonal tile, the
  // others go round.  The last ones may repeat a tile (in = false): a conditional load
  // would make the in-order wait counters conservative.
  auto upper = [&](int n, int& a, int& b) -> bool {
    if (n == 0) {
      a = b = w;
      return true;
    }
    int q = w + NW * (n - 1);
    const bool in = q < NE;
    q = in ? q : NE - 1;
    b = 1;
#pragma unroll
    for (int c = 2; c < TT; ++c) b += q >= c * (c - 1) / 2 ? 1 : 0;
    a = q - b * (b - 1) / 2;
    return in;
  };
  raw_t ar[SQ];
  auto load_a = [&](long long blk) {
#pragma unroll
    for (int n = 0; n < SQ; ++n) {
      int a, b;
      upper(n, a, b);
      ar[n] = load_raw(A + blk * NN + 16 * b * NB + 16 * a);
    }
  };
  // tiles [t0, t1) of strip w of the block's coupling
  auto load_b = [&](auto& br, long long blk, int t0, int t1) {
#pragma unroll
    for (int t = t0; t < t1; ++t) br[t - t0] = load_raw(B + blk * NN + 16 * w * NB + 16 * t);
  };
  auto put = [&](BSS_GLOBAL T* g, const tile_t& t) {
#pragma unroll
    for (int h = 0; h < I::PLANES; ++h) {
      outv_t x;
#pragma unroll
      for (int q = 0; q < I::VEC; ++q) x[q] = t[I::VEC * h + q];
      *gat<outv_t>(g + 8 * h, lcol) = x;
    }
  };

  tile_t Sl[SQ];  // S_L: this wave's upper tiles
#pragma unroll
  for (int n = 0; n < SQ; ++n) Sl[n] = Mfma<T>::zero();
  // Strip w of (-1)^i Z_i (Zn) and (-1)^i W_i (Ws): the sign of Z' = -C^T W is left out of
  // the products and put back (sg) where W leaves the registers.
  tile_t Ws[TT], Zn[TT];
  load_a(start);
  if (hasL) {  // Z_1 = B_L^T
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        Zn[t][v] = (T)*gat<const Tin>(B + (long long)(start - 1) * NN + 16 * t * NB + 16 * w,
                                      I::row(lk, v) * NB + lr);
  } else {
#pragma unroll
    for (int t = 0; t < TT; ++t) Zn[t] = Mfma<T>::zero();
  }
  // fused forward sweep: wave w carries rows 16 w.. (lane row lr)
  [[maybe_unused]] T dv = T(0), accL = T(0);
  const auto dg = gptr((T*)S.d);
  if constexpr (FWD) {
    dv = dg[(long long)start * NB + 16 * w + lr];
    if (lk == 0) Fr[16 * w + lr] = dv;
  }
#pragma unroll
  for (int n = 0; n < SQ; ++n) {
    int a, b;
    if (upper(n, a, b)) I::store(up(a, b), so, cvt(ar[n]));
  }
  // Z'(a, w) = C_a^T W_w
  auto z_tile = [&](int a) -> tile_t {
    tile_t z = Mfma<T>::zero();
#pragma unroll
    for (int t = 0; t < TT; ++t) mma16<T>(z, I::load(ct(t, a), sa), Ws[t]);
    return z;
  };
  // W strip to LDS and, with its sign f, to HBM
  auto store_w = [&](long long blk, T f) {
#pragma unroll
    for (int t = 0; t < TT; ++t) I::store(wt(t, w), so, Ws[t]);
    if (f > T(0))
      put_tiles<T, NB, TT>(W + blk * NN + 16 * w * NB, wt(0, w));
    else
      put_tiles<T, NB, TT, true>(W + blk * NN + 16 * w * NB, wt(0, w));
  };
  auto s_left = [&]() {
#pragma unroll
    for (int n = 0; n < SQ; ++n) {
      int a, b;
      if (upper(n, a, b)) {
#pragma unroll
        for (int t = 0; t < TT; ++t)
          mma16<T>(Sl[n], I::load(wt(t, a), sa), I::load(wt(t, b), so));
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  for (int e = threadIdx.x; e < 256; e += 4 * NB)
    Is[I::off(e & 15, e >> 4)] = (e & 15) == (e >> 4) ? T(1) : T(0);
  if (threadIdx.x == 0) fail = 0;
  int fail_i = len;      // first failed block of the chain (thread 0)
  float piv_run = 1.0f;  // smallest pivot ratio of the chain (wave 0)
  T sg = T(1);           // (-1)^i
  __syncthreads();

  for (int i = 0; i < len; ++i) {
    const long long blk = start + i;
    const bool last = (i == len - 1);
    const bool hasC = !last || hasR;   // block couples to a later block
    const bool late = hasL && i > 0;   // the previous block's Z', S_L are still to be done

    constexpr int DQ = (NB + 63) / 64;
    float adiag[DQ];
    if (p.pivmin && w == 0) {
#pragma unroll
      for (int h = 0; h < DQ; ++h) {
        const int j = l + 64 * h, jj = j & 15;
        adiag[h] = j < NB ? (float)up(j >> 4, j >> 4)[I::off(jj, jj)] : 1.0f;
      }
    }

    inv.windows(U + blk * NN, [&](int k) {
      if (!late || TT == 1) return;
      // The previous block's Z' and S_L, in windows in which the wave holds no diagonal
      // tile.  Up to n = 48: all of it in windows -1 and 0.  Above: half of Z' in window
      // -1 and half in window 0, what a wave missed in window 1; then W's tiles to LDS
      // over C's, and S_L in window TT-1.
      constexpr int H = OWN_W ? TT : TT / 2;
      const bool first = (k == -1 && w != 0) || (k == (OWN_W ? 0 : 1) && w == 0);
      const bool second = !OWN_W && ((k == 0 && w != 1) || (k == 1 && w == 1));
      if (first) {
#pragma unroll
        for (int a = 0; a < H; ++a) {
          Zn[a] = z_tile(a);
          __builtin_amdgcn_sched_barrier(0);
        }
        if (OWN_W) s_left();
      }
      if (second) {
#pragma unroll
        for (int a = H; a < TT; ++a) {
          Zn[a] = z_tile(a);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      if (!OWN_W && k == TT - 2) store_w(blk - 1, -sg);
    });
    raw_t br[LATE ? 1 : TT];  // the last block of the last chain has no coupling
    if (!LATE && hasC) load_b(br, blk, 0, TT);
    inv.last_window(U + blk * NN);
    if (late && !OWN_W) s_left();
    __syncthreads();
    if (threadIdx.x == 0 && fail) {
      fail_i = min(fail_i, i);
      fail = 0;
    }
    if (p.pivmin && w == 0) {
      // U_jj^2 / A_jj = 1 / (Uinv_jj^2 A_jj): the fraction of the diagonal left after
      // elimination; a failed or non-finite pivot counts as 0
      float ratio = 1.0f;
#pragma unroll
      for (int h = 0; h < DQ; ++h) {
        const int j = l + 64 * h, jj = j & 15;
        if (j < NB) {
          const float ui = (float)up(j >> 4, j >> 4)[I::off(jj, jj)];
          const float q = 1.0f / (ui * ui * adiag[h]);
          ratio = fminf(ratio, (q >= 0.0f && q <= 3.0e38f) ? q : 0.0f);
        }
      }
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) ratio = fminf(ratio, __shfl_xor(ratio, o));
      piv_run = fminf(piv_run, ratio);
    }

    // [C | W] strips, in place from the last row tile up: row r needs rows t <= r
    tile_t Cs[TT];
    if constexpr (LATE) {
      constexpr int H = (TT + 1) / 2;
#pragma unroll
      for (int h = 0; h < TT; h += H) {
        raw_t q[H];
        if (hasC) load_b(q, blk, h, h + H < TT ? h + H : TT);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < H; ++t)
          if (h + t < TT) Cs[h + t] = cvt(q[t]);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
#pragma unroll
      for (int t = 0; t < TT; ++t) Cs[t] = cvt(br[t]);
      load_a(last ? blk : blk + 1);
    }
    if constexpr (FWD) dv = dg[(last ? blk : blk + 1) * NB + 16 * w + lr];
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
    if (LATE) load_a(last ? blk : blk + 1);
    // The loads are waited for here, before the stores below: those are conditional, and a
    // wait for the loads behind them would wait for the stores as well.
#pragma unroll
    for (int n = 0; n < SQ; ++n)
#pragma unroll
      for (int h = 0; h < IP; ++h) asm volatile("" : "+v"(ar[n].p[h]));
    if constexpr (FWD) asm volatile("" : "+v"(dv));
    if (hasC) {
#pragma unroll
      for (int t = 0; t < TT; ++t) I::store(ct(t, w), so, Cs[t]);
      put_tiles<T, NB, TT>(C + blk * NN + 16 * w * NB, ct(0, w));
    }
    if (OWN_W && hasL) store_w(blk, sg);
    if constexpr (FWD) {
      // y = Uinv^T r (chain_forward1_kernel's order)
      T t0 = T(0), t1 = T(0);
#pragma unroll
      for (int t = 0; t < TT; ++t)
        if (t <= w) dot16(t0, t1, I::load(up(t, w), sa), Fr + 16 * t + 4 * lk);
      const T y = row4_sum(t0 + t1);
      if (lk == 0) {
        dg[blk * NB + 16 * w + lr] = y;
        Fy[16 * w + lr] = y;
      }
    }
    __syncthreads();  // C in LDS; Uinv read by every wave
    if constexpr (FWD) {
      // r_L += W^T y;  C^T y for the next block, or r_R after the last one
      if (hasL) {
        T t0 = T(0), t1 = T(0);
#pragma unroll
        for (int t = 0; t < TT; ++t) dot16(t0, t1, Ws[t], Fy + 16 * t + 4 * lk);
        accL += sg * row4_sum(t0 + t1);
      }
      if (!last) {
        T t0 = T(0), t1 = T(0);
#pragma unroll
        for (int t = 0; t < TT; ++t) dot16(t0, t1, Cs[t], Fy + 16 * t + 4 * lk);
        const T v = dv - row4_sum(t0 + t1);
        if (lk == 0) Fr[16 * w + lr] = v;
      } else if (hasR) {
        T t = T(0);
#pragma unroll
        for (int q = 0; q < TT; ++q)
#pragma unroll
          for (int v = 0; v < 4; ++v) t = fma(Cs[q][v], Fy[16 * q + 4 * lk + v], t);
        t = row4_sum(t);
        if (lk == 0) gptr((T*)S.rR)[(long long)sepR * NB + 16 * w + lr] = t;
      }
    }
    if (hasC) {
      // A_{i+1} -= C^T C, or S_R = C^T C after the last block
#pragma unroll
      for (int n = 0; n < SQ; ++n) {
        int a, b;
        if (upper(n, a, b)) {
          tile_t c = Mfma<T>::zero();
#pragma unroll
          for (int t = 0; t < TT; ++t)
            mma16<T>(c, I::load(ct(t, a), sa), I::load(ct(t, b), so));
          if (!last)
            I::store(up(a, b), so, cvt(ar[n]) - c);
          else
            put(gptr((T*)S.SR) + (long long)sepR * NN + 16 * b * NB + 16 * a, c);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (last && hasL) {
      if (hasR) {  // B' = -W_last^T C_last: tile (w, a) is -Z'(a, w) transposed
#pragma unroll
        for (int a = 0; a < TT; ++a) {
          const tile_t z = z_tile(a);
          const auto g = gptr((T*)S.Bn) + (long long)sepL * NN + 16 * a * NB + 16 * w;
#pragma unroll
          for (int v = 0; v < 4; ++v) *gat<T>(g, I::row(lk, v) * NB + lr) = -sg * z[v];
        }
      }
      if (!OWN_W) {
        __syncthreads();  // C read by every wave
        store_w(blk, sg);
      }
      __syncthreads();
      s_left();
    } else {
      if (TT == 1 && hasL) {
        Zn[0] = z_tile(0);
        s_left();
      }
      __syncthreads();  // A_{i+1} in LDS
    }
    if (TT > 1) forget(Zn);  // written in the next block's windows
    sg = -sg;
  }
  if (hasL) {
#pragma unroll
    for (int n = 0; n < SQ; ++n) {
      int a, b;
      if (upper(n, a, b))
        put(gptr((T*)S.SL) + (long long)sepL * NN + 16 * b * NB + 16 * a, Sl[n]);
    }
    if constexpr (FWD) {
      if (lk == 0) gptr((T*)S.rL)[(long long)sepL * NB + 16 * w + lr] = accL;
    }
  }
  // the chain's first failed block (original indices increase along a chain, so the
  // first local failure is the smallest original index) and its smallest pivot ratio
  if (threadIdx.x == 0) {
    if (fail_i < len) {
      const int blk = start + fail_i;
      atomicMin(p.info + sys, (S.orig ? S.orig[blk] : blk) + 1);
    }
    if (p.pivmin) atomicMin(p.pivmin + sys, __float_as_uint(piv_run));
  }
}

}  // namespace bss
