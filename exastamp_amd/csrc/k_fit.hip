// k_fit.hip -- the fitting loss on device tensors (fitting.py): residuals, their mean
// squares and their gradients, each in one sweep.  As elementwise tensor operations the
// loss and its backward are fourteen launches, host time of 60 us and more in a step whose
// kernels take 145 us (64 boxes of 864 atoms).  Bound by the launches there, and by the
// five arrays it touches at a million atoms.
#include "xsmd_internal.hpp"

#include <algorithm>

namespace xsmd {
namespace {

constexpr int kFitThreads = 256;
constexpr int kFitBlocks = 512;  // XS_FIT_LOSS_PARTIALS / 2

__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off);
  return v;
}

// sums over the workgroup in a fixed order; the result in thread 0
__device__ __forceinline__ double block_sum(double v, double* red)
{
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double t = 0.0;
  for (int w = 0; w < kFitThreads / 64; w++) t += red[w];
  __syncthreads();
  return t;
}

// rF = F - Ft, rE = (E - Et) / n; per workgroup the sums of their squares
__global__ void __launch_bounds__(kFitThreads) k_fit_residuals(int64_t nF, const double* __restrict__ F,
                                                               const double* __restrict__ Ft, int64_t nE,
                                                               const double* __restrict__ E,
                                                               const double* __restrict__ Et,
                                                               const double* __restrict__ n, double* __restrict__ rF,
                                                               double* __restrict__ rE, double* __restrict__ part)
{
  __shared__ double red[kFitThreads / 64];
  const int64_t i0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, step = (int64_t)gridDim.x * blockDim.x;
  double sF = 0.0, sE = 0.0;
  for (int64_t i = i0; i < nF; i += step) {
    const double d = F[i] - Ft[i];
    rF[i] = d;
    sF = fma(d, d, sF);
  }
  for (int64_t i = i0; i < nE; i += step) {
    const double d = (E[i] - Et[i]) / n[i];
    rE[i] = d;
    sE = fma(d, d, sE);
  }
  sF = block_sum(sF, red);
  sE = block_sum(sE, red);
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = sF;
    part[2 * blockIdx.x + 1] = sE;
  }
}

// mean(rF^2) + w mean(rE^2)
__global__ void __launch_bounds__(kFitThreads) k_fit_loss(int blocks, const double* __restrict__ part, double nF,
                                                          double nE, double w, double* __restrict__ loss)
{
  __shared__ double red[kFitThreads / 64];
  double sF = 0.0, sE = 0.0;
  for (int b = threadIdx.x; b < blocks; b += kFitThreads) {
    sF += part[2 * b];
    sE += part[2 * b + 1];
  }
  sF = block_sum(sF, red);
  sE = block_sum(sE, red);
  if (threadIdx.x == 0) *loss = sF / nF + w * (sE / nE);
}

// dL/dF = 2 rF / nF and dL/dE = 2 w rE / (n nE), times the incoming gradient
__global__ void __launch_bounds__(kFitThreads) k_fit_grad(int64_t nF, const double* __restrict__ rF, int64_t nE,
                                                          const double* __restrict__ rE,
                                                          const double* __restrict__ n, double cF, double cE,
                                                          const double* __restrict__ g, double* __restrict__ gF,
                                                          double* __restrict__ gE)
{
  const int64_t i0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, step = (int64_t)gridDim.x * blockDim.x;
  const double gl = *g, aF = gl * cF, aE = gl * cE;
  for (int64_t i = i0; i < nF; i += step) gF[i] = rF[i] * aF;
  for (int64_t i = i0; i < nE; i += step) gE[i] = rE[i] / n[i] * aE;
}

// makes `device` current for a launch on a caller's stream, and the caller's again after
struct DeviceGuard {
  int before = -1;
  hipError_t err;
  explicit DeviceGuard(int device)
  {
    err = hipGetDevice(&before);
    if (err == hipSuccess && before != device) err = hipSetDevice(device);
  }
  ~DeviceGuard()
  {
    if (before >= 0) (void)hipSetDevice(before);
  }
};

unsigned fit_grid(int64_t nF, int64_t nE)
{
  const int64_t n = std::max(nF, nE);
  return (unsigned)std::max<int64_t>(1, std::min<int64_t>(kFitBlocks, (n + kFitThreads - 1) / kFitThreads));
}

}  // namespace
}  // namespace xsmd

extern "C" {

xs_status xs_fit_loss_dev(int device, void* stream, int64_t nF, const double* F, const double* Ft, int64_t nE,
                          const double* E, const double* Et, const double* n, double energy_weight, double* rF,
                          double* rE, double* partials, double* loss)
{
  using namespace xsmd;
  if (nF < 1 || nE < 1 || !F || !Ft || !E || !Et || !n || !rF || !rE || !partials || !loss) return XS_E_ARG;
  static_assert(2 * kFitBlocks == XS_FIT_LOSS_PARTIALS, "two sums per workgroup");
  const DeviceGuard guard(device);
  if (guard.err != hipSuccess) return XS_E_HIP;
  const unsigned g = fit_grid(nF, nE);
  const hipStream_t s = static_cast<hipStream_t>(stream);
  k_fit_residuals<<<g, kFitThreads, 0, s>>>(nF, F, Ft, nE, E, Et, n, rF, rE, partials);
  if (hipGetLastError() != hipSuccess) return XS_E_HIP;
  k_fit_loss<<<1, kFitThreads, 0, s>>>((int)g, partials, (double)nF, (double)nE, energy_weight, loss);
  return hipGetLastError() == hipSuccess ? XS_OK : XS_E_HIP;
}

xs_status xs_fit_loss_grad_dev(int device, void* stream, int64_t nF, const double* rF, int64_t nE, const double* rE,
                               const double* n, double energy_weight, const double* g, double* gF, double* gE)
{
  using namespace xsmd;
  if (nF < 1 || nE < 1 || !rF || !rE || !n || !g || !gF || !gE) return XS_E_ARG;
  const DeviceGuard guard(device);
  if (guard.err != hipSuccess) return XS_E_HIP;
  k_fit_grad<<<fit_grid(nF, nE), kFitThreads, 0, static_cast<hipStream_t>(stream)>>>(
      nF, rF, nE, rE, n, 2.0 / (double)nF, 2.0 * energy_weight / (double)nE, g, gF, gE);
  return hipGetLastError() == hipSuccess ? XS_OK : XS_E_HIP;
}

}  // extern "C"
