// kernels_impl.hpp -- launcher definitions; included by one translation unit per
// element-type combination so the (long) template instantiations compile in parallel.
#pragma once

#include "launch.hpp"
#include "chain_factor_halves.hpp"
#include "level_kernels.hpp"

namespace bss {

template <typename Tin, typename T, int NB>
static hipError_t factor_strip(const FactorLevelArgs& a, int nchains, hipStream_t s) {
  if (a.fwd) {  // fused forward sweep: see factor_fuses_forward
    if constexpr (sizeof(T) == 4 && NB <= 96)
      hipLaunchKernelGGL((chain_factor_strip_kernel<Tin, T, NB, true>), dim3(nchains),
                         dim3(4 * NB), 0, s, a);
    else
      return hipErrorInvalidValue;
  } else {
    hipLaunchKernelGGL((chain_factor_strip_kernel<Tin, T, NB>), dim3(nchains), dim3(4 * NB), 0, s,
                       a);
  }
  return hipGetLastError();
}

// FP64 factors at n = 128 (no pivot monitor: only FP32 levels are monitored)
static inline hipError_t factor_halves128(const FactorLevelArgs& a, int nchains, hipStream_t s) {
  if (a.fwd || a.pivmin) return hipErrorInvalidValue;
  hipLaunchKernelGGL((chain_factor_halves_kernel<double, 128>), dim3(nchains), dim3(512), 0, s, a);
  return hipGetLastError();
}

template <typename Tin, typename T>
hipError_t launch_factor(int nb, const FactorLevelArgs& a, int nchains, hipStream_t s) {
  if (nchains <= 0) return hipSuccess;
  switch (nb) {
    case 16: return factor_strip<Tin, T, 16>(a, nchains, s);
    case 32: return factor_strip<Tin, T, 32>(a, nchains, s);
    case 48: return factor_strip<Tin, T, 48>(a, nchains, s);
    case 64: return factor_strip<Tin, T, 64>(a, nchains, s);
    case 96: return factor_strip<Tin, T, 96>(a, nchains, s);
    case 128:  // the strip kernel's LDS: 132 KB with FP32 factors, 262 KB with FP64
      if constexpr (sizeof(T) == 4)
        return factor_strip<Tin, T, 128>(a, nchains, s);
      else
        return factor_halves128(a, nchains, s);
    default: return hipErrorInvalidValue;
  }
}

// One right-hand side on vector FMAs; several on MFMA, in FP64 one kernel up to 4, 8 and 16
// (RhsTile; a column's bits are the same in each)
template <typename T, int NB>
static hipError_t forward_nb(const SolveLevelArgs& a, int nchains, hipStream_t s) {
  const dim3 grid(nchains), block(4 * NB);
  if (a.nrhs == 1)
    hipLaunchKernelGGL((chain_forward1_kernel<T, NB>), grid, block, 0, s, a);
  else if (sizeof(T) == 8 && a.nrhs <= 4)
    hipLaunchKernelGGL((chain_forward_kernel<T, NB, sizeof(T) == 8 ? 1 : 4>), grid, block, 0, s, a);
  else if (sizeof(T) == 8 && a.nrhs <= 8)
    hipLaunchKernelGGL((chain_forward_kernel<T, NB, sizeof(T) == 8 ? 2 : 4>), grid, block, 0, s, a);
  else
    hipLaunchKernelGGL((chain_forward_kernel<T, NB, 4>), grid, block, 0, s, a);
  return hipGetLastError();
}
template <typename T, int NB>
static hipError_t backward_nb(const SolveLevelArgs& a, int nchains, hipStream_t s) {
  const dim3 grid(nchains), block(4 * NB);
  if (a.nrhs == 1)
    hipLaunchKernelGGL((chain_backward1_kernel<T, NB>), grid, block, 0, s, a);
  else if (sizeof(T) == 8 && a.nrhs <= 4)
    hipLaunchKernelGGL((chain_backward_kernel<T, NB, sizeof(T) == 8 ? 1 : 4>), grid, block, 0, s, a);
  else if (sizeof(T) == 8 && a.nrhs <= 8)
    hipLaunchKernelGGL((chain_backward_kernel<T, NB, sizeof(T) == 8 ? 2 : 4>), grid, block, 0, s, a);
  else
    hipLaunchKernelGGL((chain_backward_kernel<T, NB, 4>), grid, block, 0, s, a);
  return hipGetLastError();
}

template <typename T>
hipError_t launch_forward(int nb, const SolveLevelArgs& a, int nchains, hipStream_t s) {
  if (nchains <= 0) return hipSuccess;
  switch (nb) {
    case 16: return forward_nb<T, 16>(a, nchains, s);
    case 32: return forward_nb<T, 32>(a, nchains, s);
    case 48: return forward_nb<T, 48>(a, nchains, s);
    case 64: return forward_nb<T, 64>(a, nchains, s);
    case 96: return forward_nb<T, 96>(a, nchains, s);
    case 128: return forward_nb<T, 128>(a, nchains, s);
    default: return hipErrorInvalidValue;
  }
}

template <typename T>
hipError_t launch_backward(int nb, const SolveLevelArgs& a, int nchains, hipStream_t s) {
  if (nchains <= 0) return hipSuccess;
  switch (nb) {
    case 16: return backward_nb<T, 16>(a, nchains, s);
    case 32: return backward_nb<T, 32>(a, nchains, s);
    case 48: return backward_nb<T, 48>(a, nchains, s);
    case 64: return backward_nb<T, 64>(a, nchains, s);
    case 96: return backward_nb<T, 96>(a, nchains, s);
    case 128: return backward_nb<T, 128>(a, nchains, s);
    default: return hipErrorInvalidValue;
  }
}

template <typename Tin, typename Ts, typename To>
hipError_t launch_assemble_diag(const SepRec* seps, const LevelSys* sys, int nb, int nsep,
                                hipStream_t s) {
  if (nsep <= 0) return hipSuccess;
  hipLaunchKernelGGL((assemble_diag_kernel<Tin, Ts, To>), dim3(nsep, nb / 16), dim3(256), 0, s,
                     seps, sys, nb);
  return hipGetLastError();
}

template <typename Ts, typename To>
hipError_t launch_assemble_rhs(const SepRec* seps, const LevelSys* sys, int nd, int nsep,
                               hipStream_t s) {
  if (nsep <= 0) return hipSuccess;
  hipLaunchKernelGGL((assemble_rhs_kernel<Ts, To>), dim3(nsep), dim3(256), 0, s, seps, sys, nd);
  return hipGetLastError();
}

template <typename Ts, typename To>
hipError_t launch_scatter_sep(const SepRec* seps, const LevelSys* sys, int nd, int nsep,
                              hipStream_t s) {
  if (nsep <= 0) return hipSuccess;
  hipLaunchKernelGGL((scatter_sep_kernel<Ts, To>), dim3(nsep), dim3(256), 0, s, seps, sys, nd);
  return hipGetLastError();
}

}  // namespace bss
