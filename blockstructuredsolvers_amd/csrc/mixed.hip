// mixed.hip -- FP64 residual / norm kernels and the refinement loop (see mixed.hpp).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <string>

#include "common.hpp"
#include "mixed.hpp"
#include "pinned_pool.hpp"
#include "residual_column.hpp"
#include "residual_tiles.hpp"

namespace bss {
namespace {

thread_local std::string g_mixed_err;
size_t al(size_t b) { return (b + 255) & ~size_t(255); }

// Combine the partial maxima: berr per (system, column).  `init` records ||d_j||;
// `mnorm` first reduces ||M||_inf from the same pass.  One kRedThreads workgroup per
// system: each thread folds every kRedThreads-th partial (eight loads in flight), then
// LDS finishes the reduction.
constexpr int kRedThreads = 1024;

__global__ void __launch_bounds__(kRedThreads)
    berr_kernel(const ResSys* __restrict__ systems, const double* __restrict__ part,
                double* __restrict__ mnorm, double* __restrict__ dnorm,
                double* __restrict__ berr, int nrhs, int init, int want_mnorm) {
  static_assert(kRedThreads % kParts == 0, "a thread keeps one partial slot");
  __shared__ double red[kRedThreads];
  const int sys = blockIdx.x, tid = threadIdx.x;
  const int g0 = systems[sys].item0, g1 = systems[sys].item1;
  // the system's partials are contiguous (item-major, kParts slots each): thread t
  // reads every kRedThreads-th value, all of slot t % kParts, coalesced
  const auto base = gptr(part) + (long long)g0 * kParts;
  const long long total = (long long)(g1 - g0) * kParts;
  double m = 0.0;
  long long i = tid;
  // the partials were just written by other CUs: issue eight loads before using any
  for (; i + 7 * kRedThreads < total; i += 8 * kRedThreads) {
    double v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = base[i + u * kRedThreads];
#pragma unroll
    for (int u = 0; u < 8; ++u) m = nmax(m, v[u]);
  }
  for (; i < total; i += kRedThreads) m = nmax(m, base[i]);
  red[tid] = m;
  __syncthreads();
  if (tid < kParts) {
    for (int k = 1; k < kRedThreads / kParts; ++k) m = nmax(m, red[tid + k * kParts]);
    red[tid] = m;
  }
  __syncthreads();
  if (tid >= 16) return;
  const double mn = want_mnorm ? red[kMnormSlot] : mnorm[sys];
  if (want_mnorm && tid == 0) mnorm[sys] = mn;
  const int c = tid;
  if (c >= nrhs) return;
  const double r = red[c], x = red[16 + c], dd = red[32 + c];
  if (init) dnorm[sys * 16 + c] = dd;
  const double den = mn * x + (init ? dd : dnorm[sys * 16 + c]);
  berr[sys * nrhs + c] = den > 0.0 ? r / den : r;
}

// blocks per residual workgroup: at least 32, and at most 256 workgroups per system.  An item
// reads one B of its neighbour, and its four waves take its rows in turn.  Mixed solves with
// resident factors, us, with 16, 32 and 64 blocks: n = 64, one system of 1024 191, 212, 260; 16
// of 300 370, 366, 415; eight of 4096 1938, 1912, 1902; n = 128, 16 right-hand sides, 16 of
// 300 2020, 1867, 2495; one of 128 670, 983, 1605.
int blocks_per_item(int N) { return std::max(32, (N + 255) / 256); }

// The first pass of a solve (x = 0, so r = d): d into the FP32 vector (the iterate is not
// written: the first residual pass takes it as zero), and the item's per-column max |d_j| (as
// both the residual and the right-hand-side maxima; the iterate maximum is 0).  Elementwise,
// with no block window: one workgroup per residual work item, kInitThreads threads.
constexpr int kInitThreads = 256;

__global__ void __launch_bounds__(kInitThreads)
    init_pass_kernel(const ResItem* __restrict__ items, const ResSys* __restrict__ systems,
                     double* __restrict__ part, int n, int nrhs, int ro_k, const int* __restrict__ skip) {
  __shared__ double red[kInitThreads / 64];
  if (skip && *skip == 0) return;  // the whole workgroup leaves (uniform)
  const ResItem it = items[blockIdx.x];
  const ResSys& S = systems[it.sys];
  const long long ND = (long long)n * nrhs;
  const auto ds = gptr(S.d);
  const auto ro = gptr(S.v[ro_k]);
  const int tid = threadIdx.x, w = wave_id(), l = lane_id();
  const int per = kInitThreads / n;  // blocks per sweep of the workgroup (n <= 128)
  double* out = part + (long long)blockIdx.x * kParts;
  for (int c = 0; c < nrhs; ++c) {
    double m = 0.0;
    for (long long j = it.b0 + tid / n; tid < per * n && j < it.b1; j += per) {
      const long long e = j * ND + (long long)c * n + tid % n;
      const double v = ds[e];
      ro[e] = (float)v;
      m = nmax(m, fabs(v));
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = nmax(m, __shfl_xor(m, o));
    if (l == 0) red[w] = m;
    __syncthreads();
    if (tid == 0) {
      double t = red[0];
      for (int k = 1; k < kInitThreads / 64; ++k) t = nmax(t, red[k]);
      out[c] = t;       // max |r_c| (r = d)
      out[16 + c] = 0;  // max |x_c|
      out[32 + c] = t;  // max |d_c|
    }
    __syncthreads();
  }
  if (tid == 0) out[kMnormSlot] = 0.0;
}

// xo_k < 0: the iterate is zero
template <int NB, bool X0>
void launch_residual_nb(const MixedState& m, int xo_k, int dx_k, int xn_k, int ro_k,
                        int want_mnorm, hipStream_t s) {
  const dim3 grid(m.nitems), block(64 * kColWaves);
  if (m.nrhs == 1 && !want_mnorm)
    hipLaunchKernelGGL((residual_column_kernel<NB, false, X0>), grid, block, 0, s, m.items,
                       m.sys_dev, m.part, xo_k, dx_k, xn_k, ro_k);
  else if (m.nrhs == 1)
    hipLaunchKernelGGL((residual_column_kernel<NB, true, X0>), grid, block, 0, s, m.items,
                       m.sys_dev, m.part, xo_k, dx_k, xn_k, ro_k);
  else if (!want_mnorm)
    hipLaunchKernelGGL((residual_tiles_kernel<NB, false, X0>), grid, block, 0, s, m.items,
                       m.sys_dev, m.part, m.nrhs, xo_k, dx_k, xn_k, ro_k);
  else
    hipLaunchKernelGGL((residual_tiles_kernel<NB, true, X0>), grid, block, 0, s, m.items,
                       m.sys_dev, m.part, m.nrhs, xo_k, dx_k, xn_k, ro_k);
}
template <int NB>
hipError_t launch_residual(const MixedState& m, bool init, int xo_k, int dx_k, int xn_k,
                           int ro_k, int want_mnorm, hipStream_t s) {
  if (init)
    hipLaunchKernelGGL(init_pass_kernel, dim3(m.nitems), dim3(kInitThreads), 0, s, m.items,
                       m.sys_dev, m.part, NB, m.nrhs, ro_k, m.init_skip);
  else if (xo_k < 0)
    launch_residual_nb<NB, true>(m, xo_k, dx_k, xn_k, ro_k, want_mnorm, s);
  else
    launch_residual_nb<NB, false>(m, xo_k, dx_k, xn_k, ro_k, want_mnorm, s);
  return hipGetLastError();
}

// profiler kinds (enum bss_kernel_kind in bss.h)
constexpr int kKindResidual = 6, kKindResidualInit = 7, kKindBerr = 8;

// One refinement pass: the residual kernel, then the per-system backward error.
hipError_t residual_prof(const MixedState& m, const MixedSolveHooks& h, bool init, int xo_k,
                         int dx_k, int xn_k, int ro_k, int want_mnorm, hipStream_t s) {
  hipError_t e;
  {
    void* scope = h.prof_begin ? h.prof_begin(h.ctx, init ? kKindResidualInit : kKindResidual, s)
                               : nullptr;
    switch (m.n) {
      case 16: e = launch_residual<16>(m, init, xo_k, dx_k, xn_k, ro_k, want_mnorm, s); break;
      case 32: e = launch_residual<32>(m, init, xo_k, dx_k, xn_k, ro_k, want_mnorm, s); break;
      case 48: e = launch_residual<48>(m, init, xo_k, dx_k, xn_k, ro_k, want_mnorm, s); break;
      case 64: e = launch_residual<64>(m, init, xo_k, dx_k, xn_k, ro_k, want_mnorm, s); break;
      case 96: e = launch_residual<96>(m, init, xo_k, dx_k, xn_k, ro_k, want_mnorm, s); break;
      case 128: e = launch_residual<128>(m, init, xo_k, dx_k, xn_k, ro_k, want_mnorm, s); break;
      default: e = hipErrorInvalidValue;
    }
    if (scope) h.prof_end(scope);
  }
  if (e != hipSuccess) return e;
  void* scope = h.prof_begin ? h.prof_begin(h.ctx, kKindBerr, s) : nullptr;
  hipLaunchKernelGGL(berr_kernel, dim3(m.nsys), dim3(kRedThreads), 0, s, m.sys_dev, m.part,
                     m.mnorm, m.dnorm, m.berr, m.nrhs, init ? 1 : 0, want_mnorm);
  e = hipGetLastError();
  if (scope) h.prof_end(scope);
  return e;
}

}  // namespace

size_t MixedState::bytes(const std::vector<int>& Ns, int n, int nrhs) {
  size_t b = 0, items = 0;
  const size_t S = Ns.size();
  size_t nd_all = 0;
  for (int N : Ns) {
    nd_all += (size_t)N * n * nrhs;
    items += (N + blocks_per_item(N) - 1) / blocks_per_item(N);
  }
  b += 2 * al(nd_all * 8) + 2 * al(nd_all * 4);
  b += al(items * sizeof(ResItem)) + al(S * sizeof(ResSys)) + al(items * kParts * 8);
  b += al(S * 8) + al(S * 16 * 8) + al(S * 16 * 8);
  if (factor_fuses_forward(n, true, nrhs)) b += al(nd_all * 8) + al(sizeof(int));
  return b;
}

int MixedState::attach(char* base, const std::vector<int>& Ns_, int n_, int nrhs_) {
  Ns = Ns_;
  n = n_;
  nrhs = nrhs_;
  nsys = (int)Ns.size();
  size_t o = 0;
  auto take = [&](size_t bytes) {
    char* p = base + o;
    o += al(bytes);
    return p;
  };
  sys_host.assign(nsys, ResSys{});
  std::vector<ResItem> it;
  // each vector set packs the systems like the caller's d (system s at the sum of the
  // earlier systems' N * n * nrhs), so the final iterate leaves in one copy
  size_t nd_all = 0;
  for (int N : Ns) nd_all += (size_t)N * n * nrhs;
  double* x0 = (double*)take(nd_all * 8);
  double* x1 = (double*)take(nd_all * 8);
  float* v0 = (float*)take(nd_all * 4);
  float* v1 = (float*)take(nd_all * 4);
  size_t od = 0;
  for (int s = 0; s < nsys; ++s) {
    const int N = Ns[s];
    const size_t nd = (size_t)N * n * nrhs;
    ResSys& r = sys_host[s];
    r.x[0] = x0 + od;
    r.x[1] = x1 + od;
    r.v[0] = v0 + od;
    r.v[1] = v1 + od;
    od += nd;
    r.N = N;
    r.item0 = (int)it.size();
    const int bpw = blocks_per_item(N);
    for (int b0 = 0; b0 < N; b0 += bpw) it.push_back({s, b0, std::min(N, b0 + bpw), 0});
    r.item1 = (int)it.size();
  }
  nitems = (int)it.size();
  items = (ResItem*)take(it.size() * sizeof(ResItem));
  sys_dev = (ResSys*)take(nsys * sizeof(ResSys));
  part = (double*)take((size_t)nitems * kParts * 8);
  mnorm = (double*)take(nsys * 8);
  dnorm = (double*)take((size_t)nsys * 16 * 8);
  berr = (double*)take((size_t)nsys * 16 * 8);
  dsnap = nullptr;
  dflag = nullptr;
  if (factor_fuses_forward(n, true, nrhs)) {
    dsnap = (double*)take(nd_all * 8);
    dflag = (int*)take(sizeof(int));
  }
  if (hipMemcpy(items, it.data(), it.size() * sizeof(ResItem), hipMemcpyHostToDevice) !=
      hipSuccess) {
    g_mixed_err = "work-item upload failed";
    return -1;
  }
  if (!host_berr &&
      !(host_berr = (double*)pinned_take((size_t)nsys * 16 * sizeof(double)))) {
    g_mixed_err = "pinned host allocation failed";
    return -1;
  }
  if (!berr_ready && hipEventCreateWithFlags(&berr_ready, hipEventDisableTiming) != hipSuccess) {
    berr_ready = nullptr;
    g_mixed_err = "event creation failed";
    return -1;
  }
  last_berr.assign((size_t)nsys * nrhs, 0.0);
  return 0;
}

int MixedState::bind(const double* A, const double* B, const double* d) {
  size_t oa = 0, ob = 0, od = 0;
  const size_t nn = (size_t)n * n, ndv = (size_t)n * nrhs;
  for (int s = 0; s < nsys; ++s) {
    const int N = Ns[s];
    sys_host[s].A = A + oa;
    sys_host[s].B = B ? B + ob : nullptr;
    sys_host[s].d = d + od;
    oa += (size_t)N * nn;
    ob += (size_t)std::max(N - 1, 0) * nn;
    od += (size_t)N * ndv;
  }
  if (hipMemcpy(sys_dev, sys_host.data(), nsys * sizeof(ResSys), hipMemcpyHostToDevice) !=
      hipSuccess) {
    g_mixed_err = "system-table upload failed";
    return -1;
  }
  return 0;
}

void MixedState::release() {
  pinned_give(host_berr);
  host_berr = nullptr;
  if (berr_ready) (void)hipEventDestroy(berr_ready);
  berr_ready = nullptr;
}

hipError_t wait_event_spin(hipEvent_t ev) {
  const auto t0 = std::chrono::steady_clock::now();
  for (;;) {
    const hipError_t q = hipEventQuery(ev);
    if (q != hipErrorNotReady) return q;
    if (std::chrono::steady_clock::now() - t0 > std::chrono::milliseconds(2))
      return hipEventSynchronize(ev);
  }
}

void mixed_after_factor(MixedState& m) { m.mnorm_stale = true; }

// below this tolerance the backward error after the first FP32 pass is not read
constexpr double kFirstCheckTol = 1e-9;

namespace {
__global__ void __launch_bounds__(256) snapshot_kernel(const ResSys* __restrict__ systems,
                                                       double* __restrict__ snap, long long n,
                                                       int* __restrict__ flag) {
  const double* __restrict__ d = systems[0].d;  // system 0 starts the packed d
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x)
    snap[i] = d[i];
  if (blockIdx.x == 0 && threadIdx.x == 0) *flag = 0;
}
}  // namespace

int mixed_snapshot_d(MixedState& m, hipStream_t s) {
  if (!m.dsnap || !m.dflag) {
    g_mixed_err = "no d snapshot in this workspace";
    return -1;
  }
  long long nd = 0;
  for (int N : m.Ns) nd += (long long)N * m.n * m.nrhs;
  const int grid = (int)std::min<long long>((nd + 255) / 256, 4096);
  hipLaunchKernelGGL(snapshot_kernel, dim3(grid), dim3(256), 0, s, m.sys_dev, m.dsnap, nd,
                     m.dflag);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    g_mixed_err = hipGetErrorString(e);
    return -1;
  }
  return 0;
}

int mixed_first_pass(MixedState& m, const MixedSolveHooks& h, hipStream_t s) {
  // x = 0, r = d (as FP32 into v[0]), ||d||.  With init_skip the kernel may leave at
  // once; the backward-error kernel after it still runs, on the partial norms the
  // skipped pass wrote the last time (nothing else writes them in between)
  const hipError_t e = residual_prof(m, h, true, -1, -1, 0, 0, 0, s);
  m.init_skip = nullptr;
  if (e != hipSuccess) {
    g_mixed_err = hipGetErrorString(e);
    return -1;
  }
  return 0;
}

namespace {
// copy the packed iterate set k into the caller's d
int write_iterate(MixedState& m, double* d, int k, hipStream_t s) {
  size_t nd_all = 0;
  for (int sy = 0; sy < m.nsys; ++sy) nd_all += (size_t)m.Ns[sy] * m.n * m.nrhs;
  const hipError_t e = hipMemcpyAsync(d, m.sys_host[0].x[k], nd_all * 8,
                                      hipMemcpyDeviceToDevice, s);
  if (e != hipSuccess) {
    g_mixed_err = hipGetErrorString(e);
    return -1;
  }
  return 0;
}

// berr to the host (one small copy, polled), into last_berr; *worst = max (NaN wins)
int read_berr(MixedState& m, hipStream_t s, double* worst) {
  hipError_t e = hipMemcpyAsync(m.host_berr, m.berr, sizeof(double) * m.nsys * m.nrhs,
                                hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = hipEventRecord(m.berr_ready, s);
  if (e == hipSuccess) e = wait_event_spin(m.berr_ready);
  if (e != hipSuccess) {
    g_mixed_err = hipGetErrorString(e);
    return -1;
  }
  double w = 0.0;
  for (int k = 0; k < m.nsys * m.nrhs; ++k) {
    const double b = m.host_berr[k];
    m.last_berr[k] = b;
    w = (b != b || w != w) ? NAN : std::max(w, b);
  }
  *worst = w;
  return 0;
}
}  // namespace

int mixed_solve(MixedState& m, const MixedSolveHooks& h, double* d, double tol, int max_iters,
                int* iters, bool* converged, bool write_unconverged, hipStream_t s,
                bool first_pass_done) {
  int cur = 0, xa = 0, it = 0;
  hipError_t e;
  *converged = false;
  *iters = 0;
  if (!first_pass_done && mixed_first_pass(m, h, s) != 0) return -1;
  bool prepared = h.prepare == nullptr;
  double prev = HUGE_VAL;  // backward error at the previous check
  while (true) {
    if (h.solve32(h.ctx, cur, s) != 0) {
      g_mixed_err = "FP32 solve failed";
      return -1;
    }
    if (!prepared) {
      // the first solve is queued before the caller's check; a changed solve path
      // redoes it (d is untouched until the end, so the x = 0 pass rebuilds r = d)
      prepared = true;
      const int pr = h.prepare(h.ctx, s);
      if (pr == 1) {
        if (mixed_first_pass(m, h, s) != 0) return -1;
        if (h.solve32(h.ctx, cur, s) != 0) {
          g_mixed_err = "FP32 solve failed";
          return -1;
        }
      } else if (pr == 2) {
        // an FP32 pivot failed: every iterate would be NaN
        for (double& b : m.last_berr) b = NAN;
        return 0;
      } else if (pr != 0) {
        g_mixed_err = "solve preparation failed";
        return -1;
      }
    }
    const int want_mnorm = m.mnorm_stale ? 1 : 0;
    e = residual_prof(m, h, false, it == 0 ? -1 : xa, cur, 1 - xa, 1 - cur, want_mnorm, s);
    m.mnorm_stale = false;
    if (e != hipSuccess) {
      g_mixed_err = hipGetErrorString(e);
      return -1;
    }
    xa = 1 - xa;
    cur = 1 - cur;
    ++it;
    // One FP32 solve of d cannot reach a tolerance far below FP32's precision, so the
    // first pass is not checked: the host queues the next correction while the device
    // is still busy instead of waiting for the backward error (an exactly solvable
    // system then takes one more, harmless, correction).
    if (it == 1 && tol < kFirstCheckTol && max_iters > 1) continue;
    double worst;
    if (read_berr(m, s, &worst) != 0) return -1;
    if (worst <= tol) {
      *converged = true;
      break;
    }
    // stop short: NaN (never compares), the iteration cap, or stagnation -- refinement
    // with a contraction factor above 1/2 is not going to reach the target soon, and
    // above 1 it diverges
    if (worst != worst || it >= max_iters || !(worst <= 0.5 * prev)) break;
    prev = worst;
  }
  *iters = it;
  // the final iterate into the caller's d (the iterate set is packed like d)
  if ((*converged || write_unconverged) && write_iterate(m, d, xa, s) != 0) return -1;
  return 0;
}

int mixed_measure(MixedState& m, const MixedSolveHooks& h, hipStream_t s, double* worst) {
  size_t nd_all = 0;
  for (int sy = 0; sy < m.nsys; ++sy) nd_all += (size_t)m.Ns[sy] * m.n * m.nrhs;
  // a zero FP32 correction in set 0, then x_1 = x_0 + 0 and r = d - M x_0
  hipError_t e = hipMemsetAsync(m.sys_host[0].v[0], 0, nd_all * 4, s);
  if (e == hipSuccess) e = residual_prof(m, h, false, 0, 0, 1, 1, m.mnorm_stale ? 1 : 0, s);
  m.mnorm_stale = false;
  if (e != hipSuccess) {
    g_mixed_err = hipGetErrorString(e);
    return -1;
  }
  return read_berr(m, s, worst);
}

const char* mixed_last_error() { return g_mixed_err.c_str(); }

}  // namespace bss
