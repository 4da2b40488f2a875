// chain_factor.hpp -- fused per-chain factorisation of one recursion level: the algorithm
// and the pieces its two kernels share (chain_factor_strip.hpp; chain_factor_halves.hpp
// for FP64 factors at n = 128).
//
// A level holds N diagonal blocks A_i and N-1 couplings B_i (M = tridiag(B^T, A, B)).
// The schedule splits it into chains of consecutive interior blocks separated by
// single separator blocks.  For a chain [s .. s+m-1] with left separator L = s-1 and
// right separator R = s+m (either may be absent) the kernel eliminates the chain in
// order, keeping the fill that the left separator creates ("panel" Z):
//
//   Z_s = B_L^T,  for i = s .. s+m-1:
//     A_i  <- A_i - C_{i-1}^T C_{i-1}               (Schur update, MFMA)
//     U_i^T U_i = A_i ; Uinv_i = U_i^{-1}           (blocked potrf + inverse)
//     [C_i | W_i] = Uinv_i^T [B_i | Z_i]            (trsm as MFMA products)
//     Z_{i+1} = -C_i^T W_i ;  S_L += W_i^T W_i      (MFMA)
//   reduced system: A'_L -= S_L, A'_R -= C_last^T C_last, B'_{L,R} = -W_last^T C_last
//
// This is the reference's per-level work -- cholesky_factorize_batched! (factor the
// P-1 interior chains, src/backbone_rocm.jl:62-82), cholesky_solve_batched! with the
// 2n-column G (src/backbone_rocm.jl:84-120) and compute_schur_complement!
// (src/backbone_rocm.jl:122-138) -- re-derived so that only the one-sided panel
// W = U^{-T} G is formed (G is non-zero only in the first and last interior block,
// src/gpu_batched.jl:214-215) and the Schur complement G^T T^{-1} G = W^T W is
// accumulated as the chain is eliminated, in one launch per level with the blocks
// held in LDS.
//
// Stored factors (consumed by the substitution sweeps): Uinv_i (upper 16x16 tiles of
// the A slot), C_i (the B slot), W_i (panel slot, only for chains with a left
// separator).  One workgroup per chain; blockIdx.y is the system in a batch.
#pragma once

#include "common.hpp"
#include "plan_tables.hpp"

namespace bss {

struct FactorLevelArgs {
  const ChainRec* chains;  // one workgroup per chain
  const LevelSys* sys;     // per-system buffers of this level
  int* info;               // per system, atomicMin of the 1-based failing block index
  unsigned* pivmin;        // per system, atomicMin of the float bits of min_j U_jj^2 / A_jj
                           // over the level's blocks (null: not monitored)
  int fwd = 0;             // 1: also run this level's forward sweep for one right-hand
                           // side (chain_forward1_kernel's arithmetic, on the factors
                           // while they are on chip): d <- y in place, r_R and r_L out
                           // (chain_factor_strip_kernel only; see factor_fuses_forward)
};

template <typename T>
struct LdsPad {
  static constexpr int value = sizeof(T) == 8 ? 2 : 4;  // 16-byte column shift
};

__device__ __host__ constexpr int tile_off(int r, int c, int ld) { return 16 * c * ld + 16 * r; }

// The value of x, hidden from the optimiser: offsets derived from it are recomputed
// where they are used instead of being hoisted out of a kernel's block loop and held in
// registers for the whole chain.
__device__ inline int opaque_v(int x) {
  asm volatile("" : "+v"(x));
  return x;
}

// Cross-lane helpers for the diagonal-tile routine.
template <typename T>
__device__ inline T read_lane(T x, int lane);
template <>
__device__ inline double read_lane<double>(double x, int lane) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(x), lane);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(x), lane);
  return __hiloint2double(hi, lo);
}
template <>
__device__ inline float read_lane<float>(float x, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), lane));
}

// every lane takes the value of lane J of its 16-lane row (DPP row_newbcast; a
// broadcast never reads outside the row, so bound_ctrl changes nothing).  The FP64 form
// is one 64-bit DPP move (gfx950 has row_newbcast for 64-bit operands), not two 32-bit
// halves that each need a zeroed destination first.
template <int J>
__device__ inline double row_bcast(double x) {
  return __longlong_as_double(
      __builtin_amdgcn_mov_dpp(__double_as_longlong(x), 0x150 + J, 0xf, 0xf, true));
}
template <int J>
__device__ inline float row_bcast(float x) {
  return __int_as_float(
      __builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x150 + J, 0xf, 0xf, false));
}

// 1/sqrt(p) on the serial path, avoiding the long correctly-rounded sqrt + divide
// sequences: f64 refines the hardware estimate (about 2^-24) with one third-order step,
// y (1 + e/2 + 3 e^2/8) with e = 1 - p y^2, whose e^3 term is below rounding: four
// dependent operations where two Newton steps take eight (a 16x16 diagonal tile 3,020 ->
// 2,830 cycles, its inverse's relative error 1.6e-16 -> 1.0e-16); f32 takes v_rsq_f32 as
// is (1 ulp), the FP32 factor's own rounding level (a Newton step there measured 2% of
// the FP32 factor time and no accuracy change in the refined result).
__device__ inline double rsqrt_nr(double p) {
  const double y = __builtin_amdgcn_rsq(p);
  const double e = fma(-(p * y), y, 1.0);
  return fma(y * e, fma(e, 0.375, 0.5), y);
}
__device__ inline float rsqrt_nr(float p) { return __builtin_amdgcn_rsqf(p); }

// One elimination step J of the 16x16 tile (see diag_chol_inv16).  Lane c (of every
// 16-lane row; the four rows compute the same thing) holds column c: a[r] = A[r][c],
// e[r] = E[r][c].  Everything the step needs is in the lane's own registers or in
// lane J of the same row, so the serial path uses only readlane/DPP and VALU ops.
// `s` = 1/sqrt of pivot J.  Row J+1 is updated first: it holds the next pivot, whose
// 1/sqrt (the long dependent part of a step) then overlaps this step's other rows.
template <typename T, int J>
__device__ __attribute__((always_inline)) inline void diag_step(T (&a)[16], T (&e)[16], T s,
                                                                bool& ok) {
  // keep steps apart in the schedule: interleaving whole steps multiplies the live
  // registers (the pivot of step J+1 is already computed inside step J)
  __builtin_amdgcn_sched_barrier(0);
  const T ujc = a[J] * s;  // U[J][c]
  const T ejc = e[J] * s;  // row J of E, scaled
  a[J] = ujc;
  e[J] = ejc;
  T s_next = T(0);
  // U[J][r] = A[J][r] s = A[r][J] s (the trailing matrix stays symmetric): lane J's a[r].
  // FP32 folds the broadcast into the multiply by s (v_mul_f32 takes a DPP operand, the
  // FP64 multiply does not): 3 VALU ops per row.  FP64 moves s into the pivot-row
  // factors once per step instead, so a row costs one 64-bit DPP move and two FMAs.
  [[maybe_unused]] const T nu = -(ujc * s), ne = -(ejc * s);
  auto update = [&](int r) {
    if constexpr (sizeof(T) == 4) {
      const T ujr = row_bcast<J>(a[r]) * s;
      a[r] -= ujr * ujc;
      e[r] -= ujr * ejc;
    } else {
      const T m = row_bcast<J>(a[r]);
      e[r] = fma(m, ne, e[r]);
      a[r] = fma(m, nu, a[r]);
    }
  };
  if constexpr (J < 15) {
    update(J + 1);
    const T p = read_lane(a[J + 1], J + 1);  // pivot A[J+1][J+1]
    ok = ok && (p > T(0));
    s_next = rsqrt_nr(p);
  }
#pragma unroll
  for (int r = J + 2; r < 16; ++r) update(r);
  // E is consumed only by the final store; without this the compiler defers all of
  // its updates to the end and keeps every multiplier of every step live
#pragma unroll
  for (int r = 0; r < 16; ++r) asm volatile("" : "+v"(e[r]));
  if constexpr (J < 15) diag_step<T, J + 1>(a, e, s_next, ok);
}

// Wave-level Cholesky + inverse of one 16x16 SPD tile held (upper triangle) in LDS, with A
// and E in separate registers (the probe of tests/gpu_probe; the kernels use diag_img).
// Row operations are applied to [A | I]; at the end the right half is E = U^{-T}.
// Writes Uinv = E^T into the upper triangle of the output tile (strict lower part
// exact zeros).  Returns false if a pivot was not positive.
// OPQ: the lane's 16 load offsets are recomputed per call, not held across the caller's
// loop (for kernels whose registers are otherwise exhausted)
template <typename T, bool OPQ = false>
__device__ __attribute__((always_inline)) inline bool diag_chol_inv16(const T* at, int lda, T* ut, int ldu) {
  const int c = OPQ ? opaque_v(lane_id() & 15) : lane_id() & 15;
  T a[16], e[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    a[r] = (r <= c) ? at[c * lda + r] : at[r * lda + c];
    e[r] = (r == c) ? T(1) : T(0);
  }
  const T p0 = read_lane(a[0], 0);
  bool ok = p0 > T(0);
  diag_step<T, 0>(a, e, rsqrt_nr(p0), ok);
  if (lane_id() < 16) {
#pragma unroll
    for (int r = 0; r < 16; ++r) ut[r * ldu + c] = e[r];  // Uinv[c][r] = E[r][c]
  }
  return ok;
}

}  // namespace bss
