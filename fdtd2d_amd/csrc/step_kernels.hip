// step_kernels.hip - single-grid launches of the step kernels (interior and
// CPML-class kernels on two streams, or one fused kernel: fused_kernels.hip)
// and the RC cutoff reduction kernel. The device code is in step_device.h.
#include <hip/hip_runtime.h>

#include "step_device.h"

namespace fdtd2d {
namespace {

// RC cutoff lines for the t steps of one launch. Dev_FindMax keeps a value
// only when a later one is strictly greater, so the maximum is the largest
// value of row 0 and rows jcut .. ny-3 that is not a NaN, and a NaN at row 0
// stays; the scan (j from ny-3 down while |Ez| < edge) stops at the largest
// j >= 1 whose |Ez| is not below the edge, else at 0. Only the edge level
// carries from step to step: two waves per step find the launch's maxima side
// by side, one thread runs the edge through them, the waves scan. A wave has
// the first kAhead rows of its scan, and of its maximum, in flight together
// (clamped rows repeat one that counts anyway): the kernel is latency, 21
// work-groups. (Step by step, two block reductions each, a line took 79 us per
// 8-step launch at 3000 rows behind a step kernel of 40; side by side with
// eight loads in flight 14.6; now 7.1.)
__global__ void __launch_bounds__(128 * kMaxT) rc_kernel(const RcArgs r, int n0, int t) {
  constexpr int kAhead = 24;  // 3072 rows
  __shared__ float s_max[kMaxT][2], s_first[kMaxT], s_edge[kMaxT];
  __shared__ int s_j[kMaxT][2];
  const int e = blockIdx.x, tid = threadIdx.x, lane = tid & 63, half = (tid >> 6) & 1, s = tid >> 7;
  const int ny = r.ny, at = half * 64 + lane;
  const int ncand = 1 + max(0, (ny - 2) - r.jcut), last = ny - 3;  // rows 1 .. last are scanned
  const long long slot = (n0 + s) & (kMaxT - 1);
  const float *cm = r.cap + (slot * r.nprobe + r.map[2 * e]) * ny;
  const float *cs = r.cap + (slot * r.nprobe + r.map[2 * e + 1]) * ny;
  float scan[kAhead];
  if (s < t) {
    auto cand = [&](int q) { return q <= 0 ? cm[0] : cm[r.jcut + min(q, ncand - 1) - 1]; };
    float v[kAhead];
#pragma unroll
    for (int k = 0; k < kAhead; ++k) {
      v[k] = cand(ncand == 1 ? 0 : at + 128 * k);
      scan[k] = cs[max(0, min(1 + at + 128 * k, last))];
    }
    float m = -INFINITY;
#pragma unroll
    for (int k = 0; k < kAhead; ++k) m = fmaxf(m, v[k]);
    for (int q = at + 128 * kAhead; q < ncand; q += 128) m = fmaxf(m, cand(q));
    for (int w = 32; w > 0; w >>= 1) m = fmaxf(m, __shfl_xor(m, w));
    if (lane == 0) {
      s_max[s][half] = m;
      if (half == 0) s_first[s] = cm[0];
    }
  }
  __syncthreads();
  if (tid == 0) {
    float edge = r.edge[e];
    for (int k = 0; k < t; ++k) {
      const float c0 = s_first[k];
      const float et = (c0 != c0 ? c0 : fmaxf(s_max[k][0], s_max[k][1])) * r.level;
      if (et > edge) edge = et;
      s_edge[k] = edge;
    }
    r.edge[e] = edge;
  }
  __syncthreads();
  if (s < t) {
    const float edge = s_edge[s];
    int bj = 0;
#pragma unroll
    for (int k = 0; k < kAhead; ++k) {
      const int j = 1 + at + 128 * k;
      if (j <= last && !(fabsf(scan[k]) < edge)) bj = j;  // j grows: the last one is the largest
    }
    for (int j = 1 + at + 128 * kAhead; j <= last; j += 128)
      if (!(fabsf(cs[j]) < edge)) bj = j;
    for (int w = 32; w > 0; w >>= 1) bj = max(bj, __shfl_xor(bj, w));
    if (lane == 0) s_j[s][half] = bj;
  }
  __syncthreads();
  if (tid < t) r.spd[static_cast<long long>(n0 + 1 + tid) * r.nrc + e] = max(s_j[tid][0], s_j[tid][1]);
}

template <int T, int C, int D, int MODE>
hipError_t launch_tcd(const StepArgs &a, int src, int n0, hipStream_t s) {
  const int grid = a.n_wg[(MODE == 1 || MODE == 3) ? 1 : 0];
  if (grid == 0) return hipSuccess;
  if (a.medium_kind == kTable)
    hipLaunchKernelGGL((step_kernel<T, C, D, kTable, MODE>), dim3(grid), dim3(64 * kWavesPerWG), 0, s, a, src, n0);
  else
    hipLaunchKernelGGL((step_kernel<T, C, D, kDensity, MODE>), dim3(grid), dim3(64 * kWavesPerWG), 0, s, a, src,
                       n0);
  return hipGetLastError();
}

template <int C, int D, int MODE>
hipError_t launch_cd(const StepArgs &a, int T, int src, int n0, hipStream_t s) {
  switch (T) {
    case 1: return launch_tcd<1, C, D, MODE>(a, src, n0, s);
    case 2: return launch_tcd<2, C, D, MODE>(a, src, n0, s);
    case 3: return launch_tcd<3, C, D, MODE>(a, src, n0, s);
    case 4: return launch_tcd<4, C, D, MODE>(a, src, n0, s);
    case 5: return launch_tcd<5, C, D, MODE>(a, src, n0, s);
    case 6: return launch_tcd<6, C, D, MODE>(a, src, n0, s);
    case 7: return launch_tcd<7, C, D, MODE>(a, src, n0, s);
    case 8: return launch_tcd<8, C, D, MODE>(a, src, n0, s);
  }
  return hipErrorInvalidValue;
}

}  // namespace

hipError_t launch_rc(const RcArgs &r, int n0, int t, hipStream_t stream) {
  if (r.nrc <= 0 || t <= 0) return hipSuccess;
  if (t > kMaxT) return hipErrorInvalidValue;
  hipLaunchKernelGGL(rc_kernel, dim3(r.nrc), dim3(128 * kMaxT), 0, stream, r, n0, t);
  return hipGetLastError();
}

hipError_t launch_step(const StepArgs &a, int cls, int T, int C, int D, int src, int n0, hipStream_t stream) {
  // CPML-class work-groups always run one column per lane with the shallow
  // prefetch (their state already fills the register file); interior ones
  // take the requested shape.
  if (cls == 1) return launch_cd<1, 1, 1>(a, T, src, n0, stream);
  if (cls == 2) return launch_cd<1, 1, 3>(a, T, src, n0, stream);
  switch (C * 16 + D) {
    case 1 * 16 + 1: return launch_cd<1, 1, 0>(a, T, src, n0, stream);
    case 1 * 16 + 2: return launch_cd<1, 2, 0>(a, T, src, n0, stream);
    case 1 * 16 + 4: return launch_cd<1, 4, 0>(a, T, src, n0, stream);
    case 2 * 16 + 1: return launch_cd<2, 1, 0>(a, T, src, n0, stream);
    case 2 * 16 + 2: return launch_cd<2, 2, 0>(a, T, src, n0, stream);
    case 4 * 16 + 1: return launch_cd<4, 1, 0>(a, T, src, n0, stream);
  }
  return hipErrorInvalidValue;
}

}  // namespace fdtd2d
