// chain_solve.hpp -- per-chain forward and backward substitution sweeps of one level.
//
// With the factors of chain_factor.hpp the level's solve is, per chain,
//   forward : y_i = Uinv_i^T (d_i - C_{i-1}^T y_{i-1})          (first block: no C term)
//             r_R = C_last^T y_last,   r_L = sum_i W_i^T y_i     (reduced right-hand side)
//   [reduced system over the separators solved by the next level: x_sep]
//   backward: x_i = Uinv_i (y_i - C_i x_{i+1} - W_i x_L),  x_{last+1} = x_R
// which replaces the reference's compute_schur_RHS! (src/backbone_rocm.jl:140-154),
// update_boundary! (src/backbone_rocm.jl:156-170) and cholesky_solve_batched! with
// nd = 1 (src/backbone_rocm.jl:84-120).  Each wave owns one 16-row tile of the block.
// One right-hand side is vector FMAs; several (up to 16) are MFMA products (RhsTile).
// Factor blocks are read straight from HBM into registers, a block ahead; only the vectors
// live in LDS.
#pragma once

#include <type_traits>

#include "common.hpp"
#include "plan_tables.hpp"

namespace bss {

struct SolveLevelArgs {
  const ChainRec* chains;
  const LevelSys* sys;  // U, C, W, d; forward writes rR/rL, backward reads dn (x_sep)
  int nrhs;
  // forward sweeps: when set and *skip == 0, the sweep already ran (inside the factor
  // kernel, on the same right-hand side) and the launch does nothing
  const int* skip = nullptr;
};

template <typename T>
struct VecPad {
  static constexpr int value = sizeof(T) == 8 ? 2 : 4;
};

// zero an LDS vector buffer (NB rows x COLS columns, leading dimension LDV)
template <typename T, int LDV, int COLS, int NT>
__device__ inline void zero_vec(T* v) {
  for (int i = threadIdx.x; i < COLS * LDV; i += NT) v[i] = T(0);
}

// A tile of 16 rows and up to 4 G right-hand sides, as the sweeps' products leave it.  A
// product's operands are x, lane (row lr, k slot lk) of the matrix, and y, lane (right-hand
// side, the same k).
//   FP64, G = 1 and 2: 4x4x4 MFMAs, four blocks of four rows each, one per four right-hand
// sides: element q of a lane is row 4 (lr / 4) + lk of right-hand side 4 q + lr % 4.  They
// take a quarter of a 16x16x4's time, which a lone chain of a few right-hand sides waits for
// (three, n = 32: 2.2 -> 1.3 us a block, both sweeps; n = 128: 15.5 -> 7.4).
//   FP64, G = 4: one 16x16x4 MFMA (the same sums) with the matrix as second operand: row lr
// of right-hand side 4 q + lk, so that 16 lanes have 16 consecutive rows of d.
//   FP32: one 16x16x4 MFMA for any number: row 4 lk + q of right-hand side lr.  (4x4x1 MFMAs
// leave sums over lk to the vector unit: three right-hand sides at n = 48 were faster, 1.98
// -> 1.50 us, sixteen slower, 1.98 -> 2.74, and a column's bits must not depend on how many
// there are.)
template <typename T, int G>
struct RhsTile {
  static constexpr bool NARROW = sizeof(T) == 8 && G < 4;
  typedef std::conditional_t<sizeof(T) == 8, std::conditional_t<NARROW, double, d4_t>, f4_t> acc_t;
  static constexpr int N = NARROW ? G : 4, ACCS = NARROW ? G : 1;
  acc_t c[ACCS];
  __device__ inline void clear() {
#pragma unroll
    for (auto& x : c) x = {};
  }
  __device__ inline T get(int q) const {
    if constexpr (NARROW) return c[q];
    else return c[0][q];
  }
  __device__ inline void set(int q, T x) {
    if constexpr (NARROW) c[q] = x;
    else c[0][q] = x;
  }
  // += x y, y(g) the lane's element of its right-hand side (side()) of group g
  static __device__ inline int side() { return lane_id() & (NARROW ? 3 : 15); }
  template <typename Y>
  __device__ __attribute__((always_inline)) inline void mma(T x, Y y) {
    if constexpr (NARROW) {
#pragma unroll
      for (int g = 0; g < G; ++g) c[g] = __builtin_amdgcn_mfma_f64_4x4x4f64(x, y(g), c[g], 0, 0, 0);
    } else if constexpr (sizeof(T) == 8) {
      c[0] = Mfma<T>::mma(y(0), x, c[0]);
    } else {
      c[0] = Mfma<T>::mma(x, y(0), c[0]);
    }
  }
};
// right-hand side and row of element q
template <typename T, int G>
struct RhsLane {
  int lr, lk;
  __device__ inline RhsLane() : lr(lane_id() & 15), lk(lane_id() >> 4) {}
  __device__ inline int col(int q) const {
    return RhsTile<T, G>::NARROW ? 4 * q + (lr & 3) : sizeof(T) == 8 ? 4 * q + lk : lr;
  }
  __device__ inline int row(int q) const {
    return RhsTile<T, G>::NARROW ? 4 * (lr >> 2) + lk : sizeof(T) == 8 ? lr : 4 * lk + q;
  }
};
// d-tile (rows 16w..) from a global n x nrhs column-major block
// Every lane loads (columns past nrhs read column 0): a predicated load would make the
// in-order wait counters conservative for every later load.  load_rhs_raw leaves those
// columns as loaded, so a tile loaded ahead is not waited for until mask_rhs uses it.
template <typename T, int NB, int G, typename P>
__device__ inline RhsTile<T, G> load_rhs_raw(P g, int w, int nrhs) {
  const RhsLane<T, G> t;
  RhsTile<T, G> a;
#pragma unroll
  for (int q = 0; q < a.N; ++q)
    a.set(q, g[(t.col(q) < nrhs ? t.col(q) : 0) * NB + 16 * w + t.row(q)]);
  return a;
}
template <typename T, int G>
__device__ inline RhsTile<T, G> mask_rhs(RhsTile<T, G> a, int nrhs) {
  const RhsLane<T, G> t;
#pragma unroll
  for (int q = 0; q < a.N; ++q) a.set(q, t.col(q) < nrhs ? a.get(q) : T(0));
  return a;
}
template <typename T, int NB, int G, typename P>
__device__ inline RhsTile<T, G> load_rhs_tile(P g, int w, int nrhs) {
  return mask_rhs<T, G>(load_rhs_raw<T, NB, G>(g, w, nrhs), nrhs);
}
template <typename T, int NB, int G, typename P>
__device__ inline void store_rhs_tile(P g, int w, int nrhs, const RhsTile<T, G>& a) {
  const RhsLane<T, G> t;
  if constexpr (sizeof(T) == 4) {
    if (t.lr < nrhs) {
#pragma unroll
      for (int q = 0; q < a.N; ++q) g[t.lr * NB + 16 * w + t.row(q)] = a.get(q);
    }
  } else {
#pragma unroll
    for (int q = 0; q < a.N; ++q)
      if (t.col(q) < nrhs) g[t.col(q) * NB + 16 * w + t.row(q)] = a.get(q);
  }
}
// the same tile to an LDS vector buffer
template <typename T, int LDV, int G>
__device__ inline void rhs_to_lds(T* b, int w, const RhsTile<T, G>& a) {
  const RhsLane<T, G> t;
#pragma unroll
  for (int q = 0; q < a.N; ++q) b[t.col(q) * LDV + 16 * w + t.row(q)] = a.get(q);
}

// global n x nrhs block -> LDS vector buffer (columns >= nrhs left untouched)
template <typename T, int NB, int LDV, int NT, typename P>
__device__ inline void load_vec(P g, T* v, int nrhs) {
  for (int i = threadIdx.x; i < NB * nrhs; i += NT) v[(i / NB) * LDV + (i % NB)] = g[i];
}

// The HBM operand of a 16-row product X y, loaded ahead into registers: rows i = 0..15 of X
// over the 16-deep k slices [s_lo, s_hi), X[i][k] at xb[k*ldx + i].
template <typename T, int NB>
struct XOps {
  T a[NB / 16][4];
  template <typename P>
  __device__ inline void load(P __restrict__ xb, int ldx, int s_lo = 0,
                              int s_hi = NB / 16) {
    const int l = lane_id();
    const int lr = l & 15, lk = l >> 4;
    // slices outside [s_lo, s_hi) re-read an in-range slice (a cache hit) and are zeroed:
    // a fixed number of loads per call keeps the in-order wait counters exact
#pragma unroll
    for (int s = 0; s < NB / 16; ++s)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int sc = s < s_lo ? s_lo : (s >= s_hi ? s_hi - 1 : s);
        const int k = 16 * sc + 4 * lk + q;
        const T x = xb[k * ldx + lr];
        a[s][q] = (s >= s_lo && s < s_hi) ? x : T(0);
      }
  }
  // acc (+/-)= X Y over the slices [s_lo, s_hi), Y[k][j] at yb[j*ldy + k] (LDS)
  template <bool NEG, int G>
  __device__ inline void mma(RhsTile<T, G>& acc, const T* __restrict__ yb, int ldy, int s_lo = 0,
                             int s_hi = NB / 16) const {
    const T* y = yb + acc.side() * ldy + 4 * (lane_id() >> 4);
#pragma unroll
    for (int s = 0; s < NB / 16; ++s) {
      if (s < s_lo || s >= s_hi) continue;
#pragma unroll
      for (int q = 0; q < 4; ++q)
        acc.mma(NEG ? -a[s][q] : a[s][q], [&](int g) { return y[4 * g * ldy + 16 * s + q]; });
    }
  }
  // One right-hand side: (X y)_i for row i = lane % 16 over the slices [s_lo, s_hi),
  // y[k] at yb[k] (LDS), in every lane of the row.  Vector FMAs over the lane's own k
  // slots, then a sum over the four lanes that share the row.
  __device__ inline T dot(const T* __restrict__ yb, int s_lo = 0, int s_hi = NB / 16) const {
    const int lk = lane_id() >> 4;
    T t0 = T(0), t1 = T(0);
#pragma unroll
    for (int s = 0; s < NB / 16; ++s) {
      if (s < s_lo || s >= s_hi) continue;
      t0 = fma(a[s][0], yb[16 * s + 4 * lk + 0], t0);
      t1 = fma(a[s][1], yb[16 * s + 4 * lk + 1], t1);
      t0 = fma(a[s][2], yb[16 * s + 4 * lk + 2], t0);
      t1 = fma(a[s][3], yb[16 * s + 4 * lk + 3], t1);
    }
    return row4_sum(t0 + t1);
  }
};

// sum over the four lanes of a quad, as (t0 + t1) + (t2 + t3), in each of them
template <int CTRL>
__device__ inline float quad_perm(float x) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), CTRL, 0xf, 0xf, true));
}
template <int CTRL>
__device__ inline double quad_perm(double x) {
  return __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(x), CTRL, 0xf, 0xf, true),
                          __builtin_amdgcn_mov_dpp(__double2loint(x), CTRL, 0xf, 0xf, true));
}
template <typename T>
__device__ inline T quad_sum(T t) {
  t += quad_perm<0xB1>(t);  // lane ^ 1
  return t + quad_perm<0x4E>(t);  // lane ^ 2
}

// The HBM operand of a product with a transposed panel, X^T y, loaded ahead: the 16
// consecutive columns of X at xb over the row slices [s_lo, s_hi).  Lane l has rows
// VEC (l % 4).. of column l / 4, so that four lanes read 64 contiguous bytes: a load of 1
// KB takes the CU's address unit 20 cycles, with a lane's column l % 16 (the order of the
// MFMA operand) 64, which bounded the sweeps wherever a CU has a chain or two.  One
// right-hand side, one chain, both sweeps: n = 64 3.67 -> 2.43 us a block in FP64, n = 128 5.81
// -> 3.18 in FP32.  MF: in the order of the MFMA operand all the same, for FP32 products up to
// n = 48, whose few loads hide behind the change of places that the other order needs.
template <typename T, int NB, bool MF = false>
struct TOps {
  static constexpr int VEC = 16 / sizeof(T), H = 4 / VEC, TT = NB / 16;
  typedef T vec_t __attribute__((ext_vector_type(VEC)));
  vec_t a[TT][H];
  template <typename P>
  __device__ inline void load(P __restrict__ xb, int s_lo = 0, int s_hi = TT) {
    const int l = lane_id();
    const auto g = MF ? xb + (l & 15) * NB + VEC * (l >> 4) : xb + (l >> 2) * NB + VEC * (l & 3);
    // slices outside [s_lo, s_hi) re-read an in-range one, as in XOps; they are not used
#pragma unroll
    for (int s = 0; s < TT; ++s) {
      const int sc = s < s_lo ? s_lo : (s >= s_hi ? s_hi - 1 : s);
#pragma unroll
      for (int h = 0; h < H; ++h) a[s][h] = *(const BSS_GLOBAL vec_t*)(g + 16 * sc + 4 * VEC * h);
    }
  }
  // One right-hand side: (X^T y) of column l / 4, in the four lanes of the quad.  FP32: the
  // order of the factor kernel's fused sweep (dot16, row4_sum).
  __device__ inline T dot(const T* __restrict__ yb, int s_lo = 0, int s_hi = TT) const {
    const T* y = yb + VEC * (lane_id() & 3);
    T t0 = T(0), t1 = T(0);
#pragma unroll
    for (int s = 0; s < TT; ++s) {
      if (s < s_lo || s >= s_hi) continue;
#pragma unroll
      for (int h = 0; h < H; ++h)
#pragma unroll
        for (int q = 0; q < VEC; q += 2) {
          t0 = fma(a[s][h][q], y[16 * s + 4 * VEC * h + q], t0);
          t1 = fma(a[s][h][q + 1], y[16 * s + 4 * VEC * h + q + 1], t1);
        }
    }
    return quad_sum(t0 + t1);
  }
  // Several: acc (+/-)= X^T Y, Y[k][j] at yb[j*ldy + k] (LDS).  The operand's lanes change
  // places through `buf` (2 H KB of this wave's LDS, two slices in turn), each quad's vectors
  // rotated by their column so that no bank is met twice.
  template <bool NEG, int G>
  __device__ inline void mma(RhsTile<T, G>& acc, const T* __restrict__ yb, int ldy, T* buf,
                             int s_lo = 0, int s_hi = TT) const {
    const int l = lane_id(), lr = l & 15, lk = l >> 4;
    [[maybe_unused]] const int put = (l & ~3) | ((l + (l >> 4)) & 3), get = 4 * lr + ((lk + (lr >> 2)) & 3);
    const T* y = yb + acc.side() * ldy + VEC * lk;
#pragma unroll
    for (int s = 0; s < TT; ++s) {
      if (s < s_lo || s >= s_hi) continue;
      [[maybe_unused]] vec_t* b = (vec_t*)buf + (s & 1) * H * 64;
      if constexpr (!MF) {
#pragma unroll
        for (int h = 0; h < H; ++h) b[64 * h + put] = a[s][h];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
        __builtin_amdgcn_wave_barrier();
      }
#pragma unroll
      for (int h = 0; h < H; ++h) {
        const vec_t x = MF ? a[s][h] : b[64 * h + get];
        vec_t z[RhsTile<T, G>::ACCS];
#pragma unroll
        for (int g = 0; g < RhsTile<T, G>::ACCS; ++g)
          z[g] = *(const vec_t*)(y + 4 * g * ldy + 16 * s + 4 * VEC * h);
#pragma unroll
        for (int q = 0; q < VEC; ++q)
          acc.mma(NEG ? -x[q] : x[q], [&](int g) { return z[g][q]; });
      }
    }
    if constexpr (!MF) {
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
      __builtin_amdgcn_wave_barrier();
    }
  }
};

// Several right-hand sides, up to 4 G.  In FP64 at n = 128 the three panels of 64 registers and
// the tiles do not quite fit: 3 registers go to scratch with G = 2, 38 (88 bytes a lane) with 4.
template <typename T, int NB, int G>
__global__ void __launch_bounds__(4 * NB) chain_forward_kernel(SolveLevelArgs p) {
  if (p.skip && *p.skip == 0) return;  // the whole workgroup leaves (uniform)
  constexpr int TT = NB / 16;
  constexpr int NT = 64 * TT;
  constexpr int LDV = NB + VecPad<T>::value;
  constexpr long long NN = (long long)NB * NB;
  typedef RhsTile<T, G> tile_t;
  constexpr bool MF = sizeof(T) == 4 && NB <= 48;
  typedef TOps<T, NB, MF> ops_t;
  __shared__ __attribute__((aligned(16))) T Y[4 * G * LDV];
  __shared__ __attribute__((aligned(16))) T R[4 * G * LDV];
  __shared__ __attribute__((aligned(16))) T turn[TT][MF ? 4 : 2 * 256];

  const ChainRec cd = p.chains[blockIdx.x];
  const int start = cd.start, len = cd.len, sepL = cd.sepL, sepR = cd.sepR;
  const LevelSys S = p.sys[cd.slot];
  const int nrhs = p.nrhs;
  const long long ND = (long long)NB * nrhs;
  const auto U = gptr((const T*)S.U);
  const auto C = gptr((const T*)S.C);
  const auto W = gptr((const T*)S.W);
  const auto d = gptr((T*)S.d);
  const int w = wave_id();
  // right-hand side of block q: below the top level (fused hand-off) it is assembled
  // from the previous level, d[q] = dp[pp[q]] - rRp[q] - rLp[q]
  const bool assemble = S.fused && S.dp;
  // the loaded parts of a right-hand side tile, combined only where the tile is used
  // (so a tile loaded one block ahead does not make this block wait for it)
  struct RhsParts {
    tile_t a, r, l;
  };
  auto rhs_parts = [&](long long q) -> RhsParts {
    RhsParts t{};
    if (!assemble) {
      t.a = load_rhs_raw<T, NB, G>(d + q * ND, w, nrhs);
    } else {
      t.a = load_rhs_raw<T, NB, G>(gptr((const T*)S.dp) + (long long)gptr(S.pp)[q] * ND, w, nrhs);
      t.r = load_rhs_raw<T, NB, G>(gptr((const T*)S.rRp) + q * ND, w, nrhs);
      t.l = load_rhs_raw<T, NB, G>(gptr((const T*)S.rLp) + q * ND, w, nrhs);
    }
    return t;
  };
  auto rhs_combine = [&](const RhsParts& t) -> tile_t {
    if (!assemble) return mask_rhs<T, G>(t.a, nrhs);
    tile_t a;
#pragma unroll
    for (int v = 0; v < a.N; ++v) a.set(v, t.a.get(v) - t.r.get(v) - t.l.get(v));
    return mask_rhs<T, G>(a, nrhs);
  };
  auto rhs_tile = [&](long long q) -> tile_t { return rhs_combine(rhs_parts(q)); };
  // the separators this chain owns get their assembled right-hand side, for the next
  // level: the one on its right, and a separator at block 0 (which has no chain on its
  // left; the reference layout starts a level with one)
  if (assemble && sepR >= 0) {
    const long long q = start + len;
    store_rhs_tile<T, NB, G>(d + q * ND, w, nrhs, rhs_tile(q));
  }
  if (assemble && sepL >= 0 && start == 1) store_rhs_tile<T, NB, G>(d, w, nrhs, rhs_tile(0));
  if (len <= 0) return;

  zero_vec<T, LDV, 4 * G, NT>(Y);
  zero_vec<T, LDV, 4 * G, NT>(R);
  __syncthreads();

  // Each HBM operand panel of block i+1 is loaded into the registers of block i's panel
  // once that panel's product has been consumed by a later instruction (so the
  // products have retired before their source registers are overwritten); the load
  // latency then hides behind the rest of block i.
  ops_t oc, ou, ow;  // C_{i-1} panel, Uinv column tiles t <= w, W_i panel
  ou.load(U + (long long)start * NN + 16 * w * NB, 0, w + 1);
  if (sepL >= 0) ow.load(W + (long long)start * NN + 16 * w * NB);
  tile_t accL;
  accL.clear();
  // the right-hand side tile of the next block is loaded one block ahead (below the
  // top level it is three dependent loads through the hand-off index)
  RhsParts rnext = rhs_parts(start);
  for (int i = 0; i < len; ++i) {
    const long long blk = start + i;
    tile_t acc = rhs_combine(rnext);
    if (i + 1 < len) rnext = rhs_parts(blk + 1);
    if (i > 0) oc.template mma<true, G>(acc, Y, LDV, turn[w]);
    rhs_to_lds<T, LDV, G>(R, w, acc);
    if (i + 1 < len) oc.load(C + blk * NN + 16 * w * NB);  // C_blk, used by row blk + 1
    // W_blk, into registers whose products (row blk - 1) retired before the C product
    // that the store above waited on
    if (sepL >= 0 && i > 0) ow.load(W + blk * NN + 16 * w * NB);
    __syncthreads();
    acc.clear();
    ou.template mma<false, G>(acc, R, LDV, turn[w], 0, w + 1);  // Uinv_blk^T r
    store_rhs_tile<T, NB, G>(d + blk * ND, w, nrhs, acc);
    rhs_to_lds<T, LDV, G>(Y, w, acc);
    if (i + 1 < len) ou.load(U + (blk + 1) * NN + 16 * w * NB, 0, w + 1);
    __syncthreads();
    if (sepL >= 0) ow.template mma<false, G>(accL, Y, LDV, turn[w]);
  }
  if (sepR >= 0) {
    const long long last = start + len - 1;
    oc.load(C + last * NN + 16 * w * NB);
    tile_t acc;
    acc.clear();
    oc.template mma<false, G>(acc, Y, LDV, turn[w]);
    store_rhs_tile<T, NB, G>(gptr((T*)S.rR) + sepR * ND, w, nrhs, acc);
  }
  if (sepL >= 0) store_rhs_tile<T, NB, G>(gptr((T*)S.rL) + sepL * ND, w, nrhs, accL);
}

// The forward sweep for one right-hand side (nrhs = 1).  Same schedule, operand loads
// and hand-off as chain_forward_kernel; the products are vector FMAs (TOps::dot), since
// an MFMA would compute four columns to keep one.  Lane l of wave w holds element 16w + l / 4
// of a block's vector.
template <typename T, int NB>
__global__ void __launch_bounds__(4 * NB) chain_forward1_kernel(SolveLevelArgs p) {
  if (p.skip && *p.skip == 0) return;  // the whole workgroup leaves (uniform)
  constexpr int TT = NB / 16;
  constexpr long long NN = (long long)NB * NB;
  __shared__ __attribute__((aligned(16))) T Y[NB];
  __shared__ __attribute__((aligned(16))) T R[NB];

  const ChainRec cd = p.chains[blockIdx.x];
  const int start = cd.start, len = cd.len, sepL = cd.sepL, sepR = cd.sepR;
  const LevelSys S = p.sys[cd.slot];
  const auto U = gptr((const T*)S.U);
  const auto C = gptr((const T*)S.C);
  const auto W = gptr((const T*)S.W);
  const auto d = gptr((T*)S.d);
  const int w = wave_id();
  const int l = lane_id();
  const int row = 16 * w + (l >> 2);
  const bool first = (l & 3) == 0;  // of the four lanes that hold an element
  const bool assemble = S.fused && S.dp;
  struct RhsParts {
    T a, r, l;
  };
  auto rhs_parts = [&](long long q) -> RhsParts {
    RhsParts t{T(0), T(0), T(0)};
    if (!assemble) {
      t.a = d[q * NB + row];
    } else {
      t.a = gptr((const T*)S.dp)[(long long)gptr(S.pp)[q] * NB + row];
      t.r = gptr((const T*)S.rRp)[q * NB + row];
      t.l = gptr((const T*)S.rLp)[q * NB + row];
    }
    return t;
  };
  auto rhs_combine = [&](const RhsParts& t) -> T { return assemble ? t.a - t.r - t.l : t.a; };
  if (assemble && sepR >= 0) {
    const long long q = start + len;
    const T v = rhs_combine(rhs_parts(q));
    if (first) d[q * NB + row] = v;
  }
  if (assemble && sepL >= 0 && start == 1) {
    const T v = rhs_combine(rhs_parts(0));
    if (first) d[row] = v;
  }
  if (len <= 0) return;

  TOps<T, NB> oc, ou, ow;  // C_{i-1} panel, Uinv column tiles t <= w, W_i panel
  ou.load(U + (long long)start * NN + 16 * w * NB, 0, w + 1);
  if (sepL >= 0) ow.load(W + (long long)start * NN + 16 * w * NB);
  T accL = T(0);
  RhsParts rnext = rhs_parts(start);
  for (int i = 0; i < len; ++i) {
    const long long blk = start + i;
    T v = rhs_combine(rnext);
    if (i + 1 < len) rnext = rhs_parts(blk + 1);
    if (i > 0) v -= oc.dot(Y);
    if (first) R[row] = v;
    if (i + 1 < len) oc.load(C + blk * NN + 16 * w * NB);
    if (sepL >= 0 && i > 0) ow.load(W + blk * NN + 16 * w * NB);
    __syncthreads();
    v = ou.dot(R, 0, w + 1);  // Uinv_blk^T r
    if (first) {
      d[blk * NB + row] = v;
      Y[row] = v;
    }
    if (i + 1 < len) ou.load(U + (blk + 1) * NN + 16 * w * NB, 0, w + 1);
    __syncthreads();
    if (sepL >= 0) accL += ow.dot(Y);
  }
  if (sepR >= 0) {
    // C_last^T y_last, straight from HBM (one use); FP32 in the fused sweep's order
    const auto cb = C + (long long)(start + len - 1) * NN + (long long)row * NB;
    T t = T(0);
#pragma unroll
    for (int s = 0; s < TT; ++s)
#pragma unroll
      for (int q = 0; q < 4; ++q) t = fma(cb[16 * s + 4 * (l & 3) + q], Y[16 * s + 4 * (l & 3) + q], t);
    t = quad_sum(t);
    if (first) gptr((T*)S.rR)[(long long)sepR * NB + row] = t;
  }
  if (sepL >= 0 && first) gptr((T*)S.rL)[(long long)sepL * NB + row] = accL;
}

// Several right-hand sides, up to 4 G.
template <typename T, int NB, int G>
__global__ void __launch_bounds__(4 * NB) chain_backward_kernel(SolveLevelArgs p) {
  constexpr int TT = NB / 16;
  constexpr int NT = 64 * TT;
  constexpr int LDV = NB + VecPad<T>::value;
  constexpr long long NN = (long long)NB * NB;
  typedef RhsTile<T, G> tile_t;
  __shared__ __attribute__((aligned(16))) T Xn[4 * G * LDV];
  __shared__ __attribute__((aligned(16))) T XL[4 * G * LDV];
  __shared__ __attribute__((aligned(16))) T R[4 * G * LDV];

  const ChainRec cd = p.chains[blockIdx.x];
  const int start = cd.start, len = cd.len, sepL = cd.sepL, sepR = cd.sepR;
  const LevelSys S = p.sys[cd.slot];
  const int nrhs = p.nrhs;
  const long long ND = (long long)NB * nrhs;
  const auto U = gptr((const T*)S.U);
  const auto C = gptr((const T*)S.C);
  const auto W = gptr((const T*)S.W);
  const auto d = gptr((T*)S.d);
  const auto xs = gptr((const T*)S.dn);
  const int w = wave_id();
  // fused hand-off: the solutions of the separators this chain owns (as in the forward
  // sweep) into this level's vector, for the level above or the caller at the top
  if (S.fused && sepR >= 0)
    store_rhs_tile<T, NB, G>(d + (long long)(start + len) * ND, w, nrhs,
                          load_rhs_tile<T, NB, G>(xs + sepR * ND, w, nrhs));
  if (S.fused && sepL >= 0 && start == 1)
    store_rhs_tile<T, NB, G>(d, w, nrhs, load_rhs_tile<T, NB, G>(xs + sepL * ND, w, nrhs));
  if (len <= 0) return;

  zero_vec<T, LDV, 4 * G, NT>(Xn);
  zero_vec<T, LDV, 4 * G, NT>(XL);
  zero_vec<T, LDV, 4 * G, NT>(R);
  __syncthreads();
  if (sepR >= 0) load_vec<T, NB, LDV, NT>(xs + sepR * ND, Xn, nrhs);
  if (sepL >= 0) load_vec<T, NB, LDV, NT>(xs + sepL * ND, XL, nrhs);
  __syncthreads();

  // operand panels of block i-1 are loaded right after block i consumed them
  XOps<T, NB> oc, ow, ou;  // rows 16w.. of C_i, W_i, and of Uinv_i (tiles t >= w)
  {
    const long long blk = start + len - 1;
    // C of the last block exists only when a right separator follows it (a level's
    // last block has no coupling block)
    if (sepR >= 0) oc.load(C + blk * NN + 16 * w, NB);
    if (sepL >= 0) ow.load(W + blk * NN + 16 * w, NB);
    ou.load(U + blk * NN + 16 * w, NB, w, TT);
  }
  tile_t rnext = load_rhs_raw<T, NB, G>(d + (long long)(start + len - 1) * ND, w, nrhs);
  for (int i = len - 1; i >= 0; --i) {
    const long long blk = start + i;
    tile_t acc = mask_rhs<T, G>(rnext, nrhs);  // y_blk; block blk - 1's tile loads one ahead
    if (i > 0) rnext = load_rhs_raw<T, NB, G>(d + (blk - 1) * ND, w, nrhs);
    if (i < len - 1 || sepR >= 0) oc.template mma<true, G>(acc, Xn, LDV);
    if (sepL >= 0) ow.template mma<true, G>(acc, XL, LDV);
    rhs_to_lds<T, LDV, G>(R, w, acc);  // consumes the products above
    if (i > 0) {
      oc.load(C + (blk - 1) * NN + 16 * w, NB);
      if (sepL >= 0) ow.load(W + (blk - 1) * NN + 16 * w, NB);
    }
    __syncthreads();
    acc.clear();
    ou.template mma<false, G>(acc, R, LDV, w, TT);  // Uinv_blk t
    store_rhs_tile<T, NB, G>(d + blk * ND, w, nrhs, acc);
    rhs_to_lds<T, LDV, G>(Xn, w, acc);
    if (i > 0) ou.load(U + (blk - 1) * NN + 16 * w, NB, w, TT);
    __syncthreads();
  }
}

// The backward sweep for one right-hand side.  Lane (lr, lk) of wave w holds element 16w + lr
// of a block's vector.
template <typename T, int NB>
__global__ void __launch_bounds__(4 * NB) chain_backward1_kernel(SolveLevelArgs p) {
  constexpr int TT = NB / 16;
  constexpr long long NN = (long long)NB * NB;
  __shared__ __attribute__((aligned(16))) T Xn[NB];
  __shared__ __attribute__((aligned(16))) T XL[NB];
  __shared__ __attribute__((aligned(16))) T R[NB];

  const ChainRec cd = p.chains[blockIdx.x];
  const int start = cd.start, len = cd.len, sepL = cd.sepL, sepR = cd.sepR;
  const LevelSys S = p.sys[cd.slot];
  const auto U = gptr((const T*)S.U);
  const auto C = gptr((const T*)S.C);
  const auto W = gptr((const T*)S.W);
  const auto d = gptr((T*)S.d);
  const auto xs = gptr((const T*)S.dn);
  const int w = wave_id();
  const int l = lane_id(), lr = l & 15, lk = l >> 4;
  const int row = 16 * w + lr;
  if (S.fused && sepR >= 0) {
    const T v = xs[(long long)sepR * NB + row];
    if (lk == 0) d[(long long)(start + len) * NB + row] = v;
  }
  if (S.fused && sepL >= 0 && start == 1) {
    const T v = xs[(long long)sepL * NB + row];
    if (lk == 0) d[row] = v;
  }
  if (len <= 0) return;

  // the separator solutions (read only when the separator exists)
  if (threadIdx.x < NB) {
    const int k = threadIdx.x;
    if (sepR >= 0) Xn[k] = xs[(long long)sepR * NB + k];
    if (sepL >= 0) XL[k] = xs[(long long)sepL * NB + k];
  }
  __syncthreads();

  XOps<T, NB> oc, ow, ou;  // rows 16w.. of C_i, W_i, and of Uinv_i (tiles t >= w)
  {
    const long long blk = start + len - 1;
    if (sepR >= 0) oc.load(C + blk * NN + 16 * w, NB);
    if (sepL >= 0) ow.load(W + blk * NN + 16 * w, NB);
    ou.load(U + blk * NN + 16 * w, NB, w, TT);
  }
  T rnext = d[(long long)(start + len - 1) * NB + row];
  for (int i = len - 1; i >= 0; --i) {
    const long long blk = start + i;
    T v = rnext;
    if (i > 0) rnext = d[(blk - 1) * NB + row];
    if (i < len - 1 || sepR >= 0) v -= oc.dot(Xn);
    if (sepL >= 0) v -= ow.dot(XL);
    if (lk == 0) R[row] = v;
    if (i > 0) {
      oc.load(C + (blk - 1) * NN + 16 * w, NB);
      if (sepL >= 0) ow.load(W + (blk - 1) * NN + 16 * w, NB);
    }
    __syncthreads();
    v = ou.dot(R, w, TT);  // Uinv_blk t
    if (lk == 0) {
      d[blk * NB + row] = v;
      Xn[row] = v;
    }
    if (i > 0) ou.load(U + (blk - 1) * NN + 16 * w, NB, w, TT);
    __syncthreads();
  }
}

}  // namespace bss
