// Traversal kernels of the wavefront path integrator: closest hits of the
// live paths (extend) and visibility of the shadow records.
#include <hip/hip_runtime.h>

#include "pt_wave.h"

namespace rrhip {
namespace {

using namespace pt;

// Profiling kernels: a wave's traversal fetches summed into prof[0..2].
// Waves without a fetch add nothing: the atomics, all on three addresses,
// were most of a profiled late round (64 rounds of a 200 x 200 cloud room:
// closest hits 23.6 -> 1.1 ms with this and the smaller grid).
__device__ __forceinline__ void add_counts(unsigned long long* prof, const TraceCount& tc) {
  uint32_t v[3] = {tc.nodes, tc.tris, tc.insts};
#pragma unroll
  for (int k = 0; k < 3; k++)
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v[k] += __shfl_xor(v[k], off);
  if ((threadIdx.x & 63u) == 0) {
#pragma unroll
    for (int k = 0; k < 3; k++)
      if (v[k]) atomicAdd(prof + k, (unsigned long long)v[k]);
  }
}

// STACK: LDS entries per lane, the smallest size >= the scene's bound
// (fewer bytes per block, more resident waves).
template <int STACK, bool MOTION, int GEO, bool COUNT = false>
__global__ __launch_bounds__(kTraceBlock) void extend_kernel(PtSceneView S, PathBuffers P, const uint32_t* __restrict__ q) {
  __shared__ uint32_t s_stack[STACK * kTraceBlock];
  uint32_t* stk = s_stack + threadIdx.x;
  const uint32_t n = P.live();
  const uint32_t stride = gridDim.x * blockDim.x;
  TraceCount tc;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    extend_one<MOTION, GEO, COUNT>(S, P, q[i], stk, &tc);
  if (COUNT) add_counts(P.prof, tc);
}

template <int STACK, bool WALK, bool MOTION, int GEO, bool COUNT = false>
__global__ __launch_bounds__(kTraceBlock) void shadow_kernel(PtSceneView S, PathBuffers P) {
  __shared__ uint32_t s_stack[STACK * kTraceBlock];
  uint32_t* stk = s_stack + threadIdx.x;
  const uint32_t n = P.shadows();
  const uint32_t stride = gridDim.x * blockDim.x;
  TraceCount tc;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    shadow_one_t<WALK, MOTION, GEO, COUNT>(S, P, i, stk, &tc);
  if (COUNT) add_counts(P.prof + 3, tc);
}

// The live paths' closest hits and the round before's shadow records in one
// launch (opaque scenes): the two do not depend on each other, and a launch
// ends with the few waves that hold its longest rays, so the shadow rays run
// under the closest hits' end instead of after it. Extension rays, the
// longer ones, come first. A wave's lanes all hold the same kind of ray.
// With the counter rotation's launch gone as well, device time a frame: 540p
// instanced field 18.6 -> 16.1 ms, 200 x 200 cloud room 4.46 -> 3.88, 256 x
// 256 box room 1.08 -> 1.02.
template <int STACK, bool MOTION, int GEO>
__global__ __launch_bounds__(kTraceBlock) void trace_kernel(PtSceneView S, PathBuffers P, const uint32_t* __restrict__ q) {
  constexpr int SG = GEO & ~kGeoSt;  // shadow rays need no texture coordinates
  __shared__ uint32_t s_stack[STACK * kTraceBlock];
  uint32_t* stk = s_stack + threadIdx.x;
  const uint32_t live = P.live(), first = (live + 63u) & ~63u, n = first + P.shadows();
  const uint32_t stride = gridDim.x * blockDim.x;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    if (i >= first)
      shadow_one_t<false, MOTION, SG>(S, P, i - first, stk);
    else if (i < live)
      extend_one<MOTION, GEO>(S, P, q[i], stk);
  }
}

// Launch of extend / shadow for the scene's stack size, transparency,
// motion and quadrics; with P.prof set, the counting variants.
template <int STACK, bool MOTION, int GEO, bool COUNT>
void launch_trace_counted(const PtSceneView& S, const PathBuffers& P, const uint32_t* q, uint32_t gt, TraceWork work,
                          hipStream_t st) {
  constexpr int SG = GEO & ~kGeoSt;  // shadow rays need texture coordinates only for a bound presence
  if (work == kTraceExtend)
    hipLaunchKernelGGL((extend_kernel<STACK, MOTION, GEO, COUNT>), dim3(gt), dim3(kTraceBlock), 0, st, S, P, q);
  else if (S.transparent && (GEO & kGeoSt) && (S.patterns & 2u))
    hipLaunchKernelGGL((shadow_kernel<STACK, true, MOTION, GEO, COUNT>), dim3(gt), dim3(kTraceBlock), 0, st, S, P);
  else if (S.transparent)
    hipLaunchKernelGGL((shadow_kernel<STACK, true, MOTION, SG, COUNT>), dim3(gt), dim3(kTraceBlock), 0, st, S, P);
  else if (work == kTraceRound)
    hipLaunchKernelGGL((trace_kernel<STACK, MOTION, GEO>), dim3(gt), dim3(kTraceBlock), 0, st, S, P, q);
  else
    hipLaunchKernelGGL((shadow_kernel<STACK, false, MOTION, SG, COUNT>), dim3(gt), dim3(kTraceBlock), 0, st, S, P);
}

template <int STACK, bool MOTION, int GEO>
void launch_trace_kernels(const PtSceneView& S, const PathBuffers& P, const uint32_t* q, uint32_t gt, TraceWork work,
                          hipStream_t st) {
  if (P.prof)
    launch_trace_counted<STACK, MOTION, GEO, true>(S, P, q, gt, work, st);
  else
    launch_trace_counted<STACK, MOTION, GEO, false>(S, P, q, gt, work, st);
}

}  // namespace

// Scenes with pattern-bound materials take full-stack extension kernels
// that also record each hit's texture coordinates, with the geometry
// classes chosen as below (their shadow rays take the kernels below).
// Scenes with loose quadrics take the full-stack kernels with the quadric
// solvers (and the curve test, for scenes with both), scenes with curve
// sets alone the kernels with the curve test only (the f64 quartic's
// registers stay out of them); one instantiation per motion flag. Every
// other scene keeps the lean kernels. Static scenes without quadrics or
// patterns take a 32-entry stack when it holds theirs: four (curves) or
// five waves per SIMD instead of three.
hipError_t pt_launch_trace(const PtSceneView& S, const PathBuffers& P, const uint32_t* q, uint32_t gt, TraceWork work,
                           hipStream_t st) {
  // only opaque scenes' unprofiled kernels hold both kinds of ray
  if (work == kTraceRound && (S.transparent || P.prof)) return hipErrorInvalidValue;
  if (work != kTraceShadow && !q) return hipErrorInvalidValue;
  const bool small = S.stack_need <= 32;
  constexpr int kAll = kGeoQuadrics | kGeoCurves;
  if (S.patterns) {  // hits also record their texture coordinates
    if (S.num_quadrics && S.motion)
      launch_trace_kernels<kTraceStack, true, kAll | kGeoSt>(S, P, q, gt, work, st);
    else if (S.num_quadrics)
      launch_trace_kernels<kTraceStack, false, kAll | kGeoSt>(S, P, q, gt, work, st);
    else if (S.curves && S.motion)
      launch_trace_kernels<kTraceStack, true, kGeoCurves | kGeoSt>(S, P, q, gt, work, st);
    else if (S.curves)
      launch_trace_kernels<kTraceStack, false, kGeoCurves | kGeoSt>(S, P, q, gt, work, st);
    else if (S.motion)
      launch_trace_kernels<kTraceStack, true, kGeoSt>(S, P, q, gt, work, st);
    else
      launch_trace_kernels<kTraceStack, false, kGeoSt>(S, P, q, gt, work, st);
  } else if (S.num_quadrics && S.motion)
    launch_trace_kernels<kTraceStack, true, kAll>(S, P, q, gt, work, st);
  else if (S.num_quadrics)
    launch_trace_kernels<kTraceStack, false, kAll>(S, P, q, gt, work, st);
  else if (S.curves && S.motion)
    launch_trace_kernels<kTraceStack, true, kGeoCurves>(S, P, q, gt, work, st);
  else if (S.curves && small)
    launch_trace_kernels<32, false, kGeoCurves>(S, P, q, gt, work, st);
  else if (S.curves)
    launch_trace_kernels<kTraceStack, false, kGeoCurves>(S, P, q, gt, work, st);
  else if (small && S.motion)
    launch_trace_kernels<32, true, 0>(S, P, q, gt, work, st);
  else if (small)
    launch_trace_kernels<32, false, 0>(S, P, q, gt, work, st);
  else if (S.motion)
    launch_trace_kernels<kTraceStack, true, 0>(S, P, q, gt, work, st);
  else
    launch_trace_kernels<kTraceStack, false, 0>(S, P, q, gt, work, st);
  return hipGetLastError();
}

}  // namespace rrhip
