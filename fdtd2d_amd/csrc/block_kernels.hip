// block_kernels.hip - launches of the block form of the step kernels (device
// code in block_device.h).
#include <hip/hip_runtime.h>

#include "block_device.h"

namespace fdtd2d {
namespace {

template <int C, int R, int RG, int W, int O>
hipError_t launch_shape(const StepArgs &a, int T, int src, int n0, hipStream_t s) {
  if (a.medium_kind == kTable)
    hipLaunchKernelGGL((block_kernel<C, R, RG, W, kTable, O>), dim3(a.n_blocks), dim3(64 * W), 0, s, a, src, n0, T);
  else
    hipLaunchKernelGGL((block_kernel<C, R, RG, W, kDensity, O>), dim3(a.n_blocks), dim3(64 * W), 0, s, a, src, n0, T);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_block(const StepArgs &a, int C, int R, int RG, int W, int T, int src, int n0, hipStream_t stream) {
  if (a.n_blocks <= 0) return hipSuccess;
  switch (((C * 16 + R) * 16 + RG) * 32 + W) {
    case ((1 * 16 + 4) * 16 + 2) * 32 + 12: return launch_shape<1, 4, 2, 12, 6>(a, T, src, n0, stream);
    case ((2 * 16 + 3) * 16 + 3) * 32 + 12: return launch_shape<2, 3, 3, 12, 5>(a, T, src, n0, stream);
    case ((1 * 16 + 8) * 16 + 4) * 32 + 8: return launch_shape<1, 8, 4, 8, 4>(a, T, src, n0, stream);
  }
  return hipErrorInvalidValue;
}

}  // namespace fdtd2d
