// Test support: the largest |fast_sigmoid(x) - exact_sigmoid(x)| over every fp32
// bit pattern x (non-finite x skipped), with the device code the routing kernels
// use. The routing fast path certifies its cuts with a bound of 2^-20 on this
// difference. 65,536 workgroups x 256 threads, 256 consecutive patterns each;
// one maximum per workgroup, reduced on the host. Likewise the largest relative error of
// the GEMM epilogues' SwiGLU, silu_mul(1, x), over a strided set of x in [-85, 88].
#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

#include "../../flashinfer_mlsys_amd/csrc/moe_common.h"
#include "../../flashinfer_mlsys_amd/csrc/moe_route_token.h"

namespace {

constexpr int kBlocks = 65536, kThreads = 256, kPerThread = 256;
static_assert((uint64_t)kBlocks * kThreads * kPerThread == (1ull << 32), "every fp32 pattern once");

__device__ void store_block_max(double m, double* __restrict__ block_max) {
  __shared__ double red[kThreads];
  red[threadIdx.x] = m;
  __syncthreads();
  for (int s = kThreads / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] = fmax(red[threadIdx.x], red[threadIdx.x + s]);
    __syncthreads();
  }
  if (threadIdx.x == 0) block_max[blockIdx.x] = red[0];
}

__global__ __launch_bounds__(kThreads) void sigmoid_bound_kernel(double* __restrict__ block_max) {
  const uint64_t first = ((uint64_t)blockIdx.x * kThreads + threadIdx.x) * kPerThread;
  double m = 0.0;
  for (int j = 0; j < kPerThread; ++j) {
    const float x = __uint_as_float((uint32_t)(first + j));
    if (!(fabsf(x) <= 3.402823466e+38f)) continue;
    m = fmax(m, fabs((double)moe::fast_sigmoid(x) - (double)moe::exact_sigmoid(x)));
  }
  store_block_max(m, block_max);
}

// Every 16th fp32 pattern.
__global__ __launch_bounds__(kThreads) void silu_bound_kernel(double* __restrict__ block_max) {
  const uint64_t first = ((uint64_t)blockIdx.x * kThreads + threadIdx.x) * kPerThread;
  double m = 0.0;
  for (int j = 0; j < kPerThread; j += 16) {
    const float x = __uint_as_float((uint32_t)(first + j) | 5u);
    if (!(x >= -85.0f && x <= 88.0f && fabsf(x) >= 1e-30f)) continue;
    const double ref = (double)x / (1.0 + exp(-(double)x));
    m = fmax(m, fabs((double)moe::silu_mul(1.0f, x) - ref) / fabs(ref));
  }
  store_block_max(m, block_max);
}

int run_blocks(void (*kernel)(double*), double* out) {
  double* d = nullptr;
  hipError_t e = hipMalloc(&d, kBlocks * sizeof(double));
  if (e != hipSuccess) return (int)e;
  hipLaunchKernelGGL(kernel, dim3(kBlocks), dim3(kThreads), 0, 0, d);
  e = hipGetLastError();
  if (e == hipSuccess) e = hipDeviceSynchronize();
  std::vector<double> h(kBlocks);
  if (e == hipSuccess) e = hipMemcpy(h.data(), d, kBlocks * sizeof(double), hipMemcpyDeviceToHost);
  (void)hipFree(d);
  if (e != hipSuccess) return (int)e;
  double m = 0.0;
  for (double v : h) m = v > m ? v : m;
  *out = m;
  return 0;
}

}  // namespace

// Each writes its maximum to *out; returns 0, or the HIP error code.
extern "C" int moe_test_fast_sigmoid_max_error(double* out) { return run_blocks(sigmoid_bound_kernel, out); }
extern "C" int moe_test_silu_max_relative_error(double* out) { return run_blocks(silu_bound_kernel, out); }
