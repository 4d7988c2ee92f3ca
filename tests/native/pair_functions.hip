// Device functions behind a C entry (built by protomol3_amd/build.py): the FP64
// functions of the pair kernel, one argument per thread, for
// tests/test_gpu_pair_functions.py, and the grid coordinate on the host, for
// tests/test_grid_coord_cpu.py.
#include <hip/hip_runtime.h>

#include "../../protomol3_amd/csrc/pmx_kernels.h"

namespace {

__global__ void k_apply(int which, int n, const double *x, double *y) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  y[i] = which == 0 ? pmx::fast_rsqrt(x[i]) : which == 1 ? pmx::fast_rcp(x[i]) : pmx::fast_exp(x[i]);
}

}  // namespace

// y = 1 / sqrt(x) (which 0), 1 / x (1), exp(x) (2) of n host values; a HIP
// error code.
extern "C" int pair_function(int which, int n, const double *x, double *y) {
  double *d = nullptr;
  hipError_t e = hipMalloc(reinterpret_cast<void **>(&d), 16 * (size_t)n);
  if (e != hipSuccess) return e;
  e = hipMemcpy(d, x, 8 * (size_t)n, hipMemcpyHostToDevice);
  if (e == hipSuccess) {
    hipLaunchKernelGGL(k_apply, dim3((n + 255) / 256), dim3(256), 0, 0, which, n, d, d + n);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipMemcpy(y, d + n, 8 * (size_t)n, hipMemcpyDeviceToHost);
  hipFree(d);
  return e;
}

extern "C" void grid_coordinate(double x, double hr, int points, int off, int *base, double *w) {
  pmx::grid_coord(x, hr, points, off, *base, *w);
}
