// smoother.hip -- block-tridiagonal normal equations of a linear state-space smoother,
// built on the device.
//
// For the model x_{i+1} = F x_i + w_i (w ~ N(0, Q)), y_i = H x_i + v_i (v ~ N(0, R))
// the smoother's normal equations are block-tridiagonal with, for every block,
//   A_i = Q^{-1} + F^T Q^{-1} F + H^T R^{-1} H,    B_i = -Q^{-1} F
// (the served-stream workload; benchmark/benchmark_kf.jl:79-154 builds the same blocks
// on the host, with A_1 and A_N special-cased, and uploads them).  Here the two n x n
// blocks are formed in FP64 and written into the reference layout (A: N blocks,
// B: N-1 blocks, column-major), so a request carries only the model matrices.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "../../include/bss.h"

namespace bss {
int api_fail(int code, const char* msg);  // records bss_last_error (bss_api.hip)
}

namespace {

constexpr int kSmootherThreads = 1024;
// Columns of a work-group (one entry a thread) and rows of a product kept in LDS at a time,
// for n <= MAXN
template <int MAXN>
struct SmootherTile {
  static constexpr int COLS = MAXN <= 32 ? 32 : kSmootherThreads / 48;
  static constexpr int KS = MAXN <= 32 ? 16 : 32, LD = KS + 1;
  double Gs[MAXN * LD];    // rows of G, one column after the other at an odd stride
  double Ps[COLS * LD];    // the same rows of S G, this work-group's columns
  double Ss[128 * KS];     // columns of S^T
  double Gc[COLS * 128];   // this work-group's columns of G

  // This thread's entry (r, c0 + cl), of nc columns from c0 on, of G^T (S G), G kk x n, S
  // kk x kk (column-major); *sg (where given) its entry of S G (kk = n).
  __device__ inline double gtsg(int n, int kk, const double* __restrict__ G,
                                const double* __restrict__ S, int c0, int nc, int r, int cl,
                                double* sg) {
    const int nt = blockDim.x;
    __syncthreads();  // the product before is done with the LDS
    for (int e = threadIdx.x; e < kk * nc; e += nt) Gc[e] = G[c0 * kk + e];
    double t = 0.0;
    for (int k0 = 0; k0 < kk; k0 += KS) {
      const int ks = min(KS, kk - k0);
      for (int e = threadIdx.x; e < KS * n; e += nt) {
        const int k = e % KS, c = e / KS;
        if (k < ks) Gs[c * LD + k] = G[c * kk + k0 + k];
      }
      for (int e = threadIdx.x; e < KS * kk; e += nt) {
        const int k = e % KS, c = e / KS;
        if (k < ks) Ss[e] = S[c * kk + k0 + k];
      }
      __syncthreads();
      for (int e = threadIdx.x; e < KS * nc; e += nt) {
        const int k = e % KS, c = e / KS;
        if (k >= ks) continue;
        double p = 0.0;
        for (int j = 0; j < kk; ++j) p += Ss[j * KS + k] * Gc[c * kk + j];
        Ps[c * LD + k] = p;
      }
      __syncthreads();
      if (cl < nc) {
        for (int k = 0; k < ks; ++k) t += Gs[r * LD + k] * Ps[cl * LD + k];
        if (sg && r >= k0 && r < k0 + ks) *sg = Ps[cl * LD + r - k0];
      }
      __syncthreads();  // the slices are read
    }
    return t;
  }
};

// A_0 and B_0 and their copies in all blocks, in one launch: a work-group forms the columns
// it has threads for (blockIdx.y) and writes them to its share of the blocks (blockIdx.x).
// A request is latency-bound: forming block 0 in a launch of its own, each entry by a double
// loop over both products, and copying it by two more took 31.5 + 4.8 + 4.0 us at n = 16,
// 300 blocks; this takes 6.4 us.  At n = 64, 128 blocks: 145 -> 22 us (53 with the products read
// from the caches entry by entry: bound by the load instructions).
// Column-major inputs: F (n x n), H (m x n), Qinv (n x n), Rinv (m x m).
template <typename T, int MAXN>
__global__ void __launch_bounds__(kSmootherThreads)
    smoother_kernel(int N, int n, int m, const double* __restrict__ F,
                    const double* __restrict__ H, const double* __restrict__ Qinv,
                    const double* __restrict__ Rinv, T* __restrict__ A, T* __restrict__ B) {
  __shared__ SmootherTile<MAXN> tile;
  const int cg = blockDim.x / n, c0 = blockIdx.y * cg, nc = min(cg, n - c0);
  const int r = threadIdx.x % n, cl = threadIdx.x / n;
  double b = 0.0;
  const double a = tile.gtsg(n, n, F, Qinv, c0, nc, r, cl, &b);
  const double h = tile.gtsg(n, m, H, Rinv, c0, nc, r, cl, nullptr);
  if (cl >= nc) return;
  const int e = (c0 + cl) * n + r;
  const T av = (T)(Qinv[e] + a + h), bv = (T)-b;
  const long long nn = (long long)n * n;
  for (long long j = blockIdx.x; j < N; j += gridDim.x) {
    A[j * nn + e] = av;
    if (j + 1 < N) B[j * nn + e] = bv;
  }
}

template <typename T>
void launch_smoother(int N, int n, int m, const double* F, const double* H, const double* Qinv,
                     const double* Rinv, T* A, T* B, hipStream_t s) {
  const int nt = std::min(n * n, kSmootherThreads), cols = nt / n, gy = (n + cols - 1) / cols;
  // (above n = 32 one work-group a CU at a time, and more would form the blocks again)
  const dim3 grid(std::min(N, (n <= 32 ? 512 : 256) / gy), gy);
  if (n <= 32)  // less LDS: two work-groups a CU
    hipLaunchKernelGGL((smoother_kernel<T, 32>), grid, dim3(nt), 0, s, N, n, m, F, H, Qinv, Rinv,
                       A, B);
  else
    hipLaunchKernelGGL((smoother_kernel<T, 128>), grid, dim3(nt), 0, s, N, n, m, F, H, Qinv,
                       Rinv, A, B);
}

}  // namespace

extern "C" int bss_build_smoother(int N, int n, int m, const double* F, const double* H,
                                  const double* Qinv, const double* Rinv, void* A, void* B,
                                  int dtype, void* stream) {
  if (N < 1 || n < 16 || n > 128 || (n % 16) != 0 || m < 1 || m > 128)
    return bss::api_fail(BSS_E_ARG, "smoother sizes: need N >= 1, n in {16, ..., 128} (multiple of 16), 1 <= m <= 128");
  if (!F || !H || !Qinv || !Rinv || !A || (N > 1 && !B))
    return bss::api_fail(BSS_E_ARG, "smoother: null buffer");
  if (dtype != BSS_F32 && dtype != BSS_F64) return bss::api_fail(BSS_E_ARG, "smoother: bad dtype");
  hipStream_t s = (hipStream_t)stream;
  if (dtype == BSS_F64)
    launch_smoother(N, n, m, F, H, Qinv, Rinv, (double*)A, (double*)B, s);
  else
    launch_smoother(N, n, m, F, H, Qinv, Rinv, (float*)A, (float*)B, s);
  return hipGetLastError() == hipSuccess ? BSS_OK : bss::api_fail(BSS_E_HIP, "smoother: launch failed");
}
