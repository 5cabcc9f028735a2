// block_kernels.hip - launches of the block form of the step kernels, for
// plans and for pools (device code in block_device.h).
#include <hip/hip_runtime.h>

#include "block_device.h"

namespace fdtd2d {
namespace {

// Calls f with the shape as constants: C, R, RG, W, the medium, and the waves
// per SIMD the registers are held to: two work-groups per CU. (For it only
// waves with events spill, up to 20 registers.)
template <class F>
hipError_t with_shape(int C, int R, int RG, int W, int medium_kind, F f) {
  const int key = ((C * 16 + R) * 16 + RG) * 16 + W;
  constexpr auto k = [](int c, int r, int rg, int w) { return ((c * 16 + r) * 16 + rg) * 16 + w; };
  const bool table = medium_kind == kTable;
  if (key == k(2, 4, 4, 12) && !table) return f.template operator()<2, 4, 4, 12, kDensity, 6>();
  if (key == k(1, 6, 3, 12)) {
    if (table) return f.template operator()<1, 6, 3, 12, kTable, 6>();
    return f.template operator()<1, 6, 3, 12, kDensity, 6>();
  }
  if (key == k(1, 4, 2, 12)) {
    if (table) return f.template operator()<1, 4, 2, 12, kTable, 6>();
    return f.template operator()<1, 4, 2, 12, kDensity, 6>();
  }
  return hipErrorInvalidValue;
}

struct PlanLaunch {
  const StepArgs &a;
  int T, src, n0;
  hipStream_t s;
  template <int C, int R, int RG, int W, int MED, int O>
  hipError_t operator()() const {
    hipLaunchKernelGGL((block_kernel<C, R, RG, W, MED, O>), dim3(a.n_blocks), dim3(64 * W), 0, s, a, src, n0, T);
    return hipGetLastError();
  }
};

struct PoolLaunch {
  const StepArgs *descs;
  const PoolQueue *q;
  int k, tp, T, grid;
  hipStream_t s;
  template <int C, int R, int RG, int W, int MED, int O>
  hipError_t operator()() const {
    hipLaunchKernelGGL((block_pool_kernel<C, R, RG, W, MED, O>), dim3(grid), dim3(64 * W), 0, s, descs, q, k, tp, T);
    return hipGetLastError();
  }
};

}  // namespace

hipError_t launch_block(const StepArgs &a, int C, int R, int RG, int W, int T, int src, int n0, hipStream_t stream) {
  if (a.n_blocks <= 0) return hipSuccess;
  return with_shape(C, R, RG, W, a.medium_kind, PlanLaunch{a, T, src, n0, stream});
}

hipError_t launch_pool_block(const StepArgs *descs, PoolQueue *q, int k, int tp, int C, int R, int RG, int W, int T,
                             int medium_kind, int grid, hipStream_t stream) {
  if (grid <= 0 || k < 0 || k >= kMaxChunk || T < 1 || T > kMaxT) return hipErrorInvalidValue;
  return with_shape(C, R, RG, W, medium_kind, PoolLaunch{descs, q, k, tp, T, grid, stream});
}

}  // namespace fdtd2d
