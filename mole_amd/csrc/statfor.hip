// Integrated autocorrelation time of every walker's local-energy series on
// the device: the estimator of scripts/statfor.rs:30-54,
//   tau = max(1, 1 + 2 sum_{i=1..min(200, n-1)} rho_i f_i),
//   rho_i = sum_{t<n-i} (x_t - m)(x_{t+i} - m) / (var (n - i)),
//   f_i = 0 from the first negative rho on, var with n - 1 (statfor.rs:86-88),
// so effective sample counts need no copy of the series to the host.
//
// tau_tile_kernel (series that fit a workgroup's LDS, from 2,048 walkers on): a
// workgroup takes 16 walkers, their series side by side in LDS; a lane takes
// one walker and 4 neighbouring lags, whose partners it slides through
// registers (two LDS reads for 4 products).  32 such lane groups make a pass of
// 128 lags, and the passes end when every walker's sum has met its first
// negative rho.  Every sum is the reference's sequential fold on one lane.
// tau_corr_kernel (the rest): one 256-thread workgroup per walker, a lag
// per thread, all lags.  Compiled with -ffp-contract=off, both results equal
// the CPU fold bit for bit.
#include <hip/hip_runtime.h>

#include "../../include/mole_gpu.h"
#include "internal.hpp"

namespace mole {

namespace {

constexpr int kTauThreads = 256;
constexpr int kTauMaxLag = 200;
constexpr int kTauLdsSamples = 8192;  // series up to this length are staged in LDS
constexpr int kTauTileMinWalkers = 2048;
constexpr int kTauTileSamples = 1000;  // 16 of them, and a pass's lags, within a CU's 160 KiB

// Bound: the serial mean and variance of a workgroup (one lane per walker),
// then FP64 issue, a multiply and an add per product.  The sum stops at the
// first negative rho, so lags past the last walker's cut are not formed: with
// all 200 lags, a thread each and two LDS reads per product, 65,536 walkers x
// 400 samples took 1,610 us a call (LDS-bound); this kernel takes 420 with 32
// groups of 4 lags (565 with 8 of 8, 455 with 16 of 8, 526 with 64 of 2: the
// fewer lags per lane, the shorter the fold that a workgroup waits for, the
// more LDS reads per product).  16 walkers per workgroup: few enough that one
// slow walker does not hold many others' lanes, and series up to 1,000 samples
// fit the LDS.
constexpr int kTileWalkers = 16, kTileStride = 17, kTilePad = 8;
constexpr int kGroups = 32, kLags = 4;

constexpr size_t tau_tile_lds(int n) {
  return sizeof(double) * ((size_t)(n + kTilePad) * kTileStride + (size_t)(kGroups * kLags + 1) * kTileWalkers);
}

__global__ void __launch_bounds__(kGroups * kTileWalkers) tau_tile_kernel(const double *trace_e, int W, size_t cap,
                                                                          size_t first, int n, double *tau_out) {
  extern __shared__ double lds[];
  double *y = lds;                                            // [n + pad][stride]
  double *corr = y + (size_t)(n + kTilePad) * kTileStride;    // [lags of a pass][walker]
  double *stat = corr + kGroups * kLags * kTileWalkers;       // the walkers' means, then their variances
  constexpr int kThreads = kGroups * kTileWalkers, kPass = kGroups * kLags;
  const int tid = threadIdx.x, wl = tid % kTileWalkers, g = tid / kTileWalkers;
  const int w0 = blockIdx.x * kTileWalkers;
  const int nw = min(kTileWalkers, W - w0);
  // kGroups consecutive samples of a walker per lane group, eight loads of a
  // lane in flight; absent walkers of the last workgroup repeat the first
  {
    const int r = tid / kGroups, t0 = tid % kGroups;
    const double *src = trace_e + (size_t)(w0 + (r < nw ? r : 0)) * cap + first;
    double *o = y + r;
    int t = t0;
    for (; t + 7 * kGroups < n; t += 8 * kGroups) {
      double v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = src[t + u * kGroups];
#pragma unroll
      for (int u = 0; u < 8; ++u) o[(t + u * kGroups) * kTileStride] = v[u];
    }
    for (; t < n; t += kGroups) o[t * kTileStride] = src[t];
  }
  for (int e = tid; e < kTilePad * kTileStride; e += kThreads) y[n * kTileStride + e] = 0.0;
  __syncthreads();
  // mean and variance: one sequential sum per walker, the next batch's reads
  // ahead of this batch's additions
  auto fold = [&](auto term) {
    const double *yt = y + tid;
    double sum = 0.0, v[8], nv[8];
    int t = 0;
    if (n >= 8) {
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = yt[u * kTileStride];
      for (; t + 8 <= n; t += 8) {
        // rows past n + pad - 1 are not read: the last batch's prefetch stays
        // within the padding
        const int tn = t + 16 <= n + kTilePad ? t + 8 : t;
#pragma unroll
        for (int u = 0; u < 8; ++u) nv[u] = yt[(tn + u) * kTileStride];
#pragma unroll
        for (int u = 0; u < 8; ++u) sum += term(v[u]);
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = nv[u];
      }
    }
    for (; t < n; ++t) sum += term(yt[t * kTileStride]);
    return sum;
  };
  if (tid < kTileWalkers) stat[tid] = fold([](double x) { return x; }) / (double)n;
  __syncthreads();
  {
    const double mean = stat[wl];
    for (int t = g; t < n; t += kGroups) y[t * kTileStride + wl] = y[t * kTileStride + wl] - mean;
  }
  __syncthreads();
  if (tid < kTileWalkers) stat[tid] = fold([](double d) { return d * d; }) / (double)(n - 1);
  __syncthreads();
  const double var = stat[wl];
  const int max_i = kTauMaxLag < n - 1 ? kTauMaxLag : n - 1;
  const double *yw = y + wl;
  double tau = 1.0;     // threads 0..15: the walker's sum
  bool done = tid >= kTileWalkers;
  for (int i0 = 0; i0 < max_i; i0 += kPass) {
    // lags b + 1 .. b + kLags of this lane; rows past n are never used
    const int b = i0 + g * kLags;
    double c[kLags], v[kLags];
#pragma unroll
    for (int j = 0; j < kLags; ++j) c[j] = 0.0;
    const int full = n - (b + kLags);  // t below it: all kLags products
    int t = 0;
    if (full >= 8) {
#pragma unroll
      for (int j = 0; j < kLags; ++j) v[j] = yw[(b + 1 + j) * kTileStride];
      for (; t + 8 <= full; t += 8) {
        double a[8], nv[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          a[u] = yw[(t + u) * kTileStride];
          nv[u] = yw[(t + u + b + 1 + kLags) * kTileStride];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
#pragma unroll
          for (int j = 0; j < kLags; ++j) {
            const double yj = u + j < kLags ? v[u + j < kLags ? u + j : 0] : nv[u + j < kLags ? 0 : u + j - kLags];
            c[j] += a[u] * yj;
          }
        }
#pragma unroll
        for (int j = 0; j < kLags; ++j) v[j] = nv[8 - kLags + j];
      }
    }
    for (; t < n - (b + 1); ++t) {
      const double a = yw[t * kTileStride];
#pragma unroll
      for (int j = 0; j < kLags; ++j)
        if (t + b + 1 + j < n) c[j] += a * yw[(t + b + 1 + j) * kTileStride];
    }
#pragma unroll
    for (int j = 0; j < kLags; ++j)
      if (b + 1 + j <= max_i) corr[(g * kLags + j) * kTileWalkers + wl] = c[j] / (var * (double)(n - (b + 1 + j)));
    __syncthreads();
    if (!done) {
      // the terms in lag order up to the first negative one (its factor f
      // and all later ones are 0; a NaN is not negative and is added)
      const int k1 = min(kPass, max_i - i0);
      for (int k = 0; k < k1; ++k) {
        const double r = corr[k * kTileWalkers + tid];
        if (r < 0.0) {
          done = true;
          break;
        }
        tau += 2.0 * r;
      }
    }
    if (__syncthreads_and(done)) break;
  }
  if (tid < nw) tau_out[w0 + tid] = tau > 1.0 ? tau : 1.0;
}

template <bool LDS>
__global__ void __launch_bounds__(kTauThreads) tau_corr_kernel(const double *trace_e, size_t cap, size_t first, int n,
                                                               double *tau_out) {
  extern __shared__ double xs[];
  __shared__ double corr[kTauMaxLag];
  __shared__ double mv[2];
  const size_t w = blockIdx.x;
  const double *src = trace_e + w * cap + first;
  const double *x = src;
  if constexpr (LDS) {
    for (int t = threadIdx.x; t < n; t += kTauThreads) xs[t] = src[t];
    __syncthreads();
    x = xs;
  }
  if (threadIdx.x == 0) {
    double mean = 0.0;
    for (int t = 0; t < n; ++t) mean += x[t];
    mean /= (double)n;
    double var = 0.0;
    for (int t = 0; t < n; ++t) var += (mean - x[t]) * (mean - x[t]);
    var /= (double)(n - 1);
    mv[0] = mean;
    mv[1] = var;
  }
  __syncthreads();
  const double mean = mv[0], var = mv[1];
  const int max_i = kTauMaxLag < n - 1 ? kTauMaxLag : n - 1;
  const int i = threadIdx.x + 1;
  if (i <= max_i) {
    double c = 0.0;
    const int m = n - i;
    int t = 0;
    // loads issued eight at a time ahead of the additions (same order)
    for (; t + 8 <= m; t += 8) {
      double a[8], b[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        a[u] = x[t + u];
        b[u] = x[t + u + i];
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) c += (a[u] - mean) * (b[u] - mean);
    }
    for (; t < m; ++t) c += (x[t] - mean) * (x[t + i] - mean);
    corr[i - 1] = c / (var * (double)m);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double tau = 1.0, f = 1.0;
    for (int k = 1; k <= max_i; ++k) {
      const double c = corr[k - 1];
      if (c < 0.0) f = 0.0;
      tau += 2.0 * c * f;
    }
    tau_out[w] = tau > 1.0 ? tau : 1.0;
  }
}

hipError_t launch_tile(const double *trace_e, int W, size_t cap, size_t first, int n, double *tau_out,
                       hipStream_t stream) {
  const size_t bytes = tau_tile_lds(n);
  if (bytes > 65536) {
    // more than the default 64 KiB of dynamic LDS needs an opt-in per kernel
    const hipError_t e = hipFuncSetAttribute((const void *)tau_tile_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                             (int)bytes);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(tau_tile_kernel, dim3((unsigned)((W + kTileWalkers - 1) / kTileWalkers)),
                     dim3(kGroups * kTileWalkers), bytes, stream, trace_e, W, cap, first, n, tau_out);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_tau_corr(const double *trace_e, int W, size_t cap, size_t first, int n, double *tau_out,
                           hipStream_t stream) {
  if (W <= 0) return hipSuccess;
  // Below 2,048 walkers a workgroup per walker has the chip to itself and its
  // lag-parallel fold is the shorter one (500 walkers x 400 samples: 52 against
  // 60 us a call; 4,096: 149 against 89).
  if (W >= kTauTileMinWalkers && n <= kTauTileSamples)
    return launch_tile(trace_e, W, cap, first, n, tau_out, stream);
  if (n <= kTauLdsSamples)
    hipLaunchKernelGGL(tau_corr_kernel<true>, dim3(W), dim3(kTauThreads), sizeof(double) * n, stream, trace_e, cap,
                       first, n, tau_out);
  else
    hipLaunchKernelGGL(tau_corr_kernel<false>, dim3(W), dim3(kTauThreads), 0, stream, trace_e, cap, first, n,
                       tau_out);
  return hipGetLastError();
}

}  // namespace mole
