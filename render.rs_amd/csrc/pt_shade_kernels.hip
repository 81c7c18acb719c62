// Shading kernels of the wavefront path integrator.
#include <hip/hip_runtime.h>

#include "pt_wave.h"

namespace rrhip {
namespace {

using namespace pt;

// Three waves per SIMD (<= 168 VGPRs): shading is latency-bound on
// scattered path-state loads, so occupancy matters more than registers.
template <bool NRC, bool TR, bool FILM = false, bool FIXED = false>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(3))) void shade_kernel(
    PtSceneView S, PathBuffers P, PtParams prm, const uint32_t* __restrict__ q, uint32_t* __restrict__ qnext,
    NrcPathBuffers N) {
  shade_pass<NRC, TR, FILM, FIXED, false>(S, P, prm, q, qnext, N);
}

// Scenes with hair fibers: the fiber BSDF's state does not fit 168
// registers next to the surface lobes', so two waves per SIMD.
template <bool TR, bool FILM, bool FIXED>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(2))) void shade_hair_kernel(
    PtSceneView S, PathBuffers P, PtParams prm, const uint32_t* __restrict__ q, uint32_t* __restrict__ qnext,
    NrcPathBuffers N) {
  shade_pass<false, TR, FILM, FIXED, true>(S, P, prm, q, qnext, N);
}

// Scenes with pattern-bound materials (and hair fibers, if any): the
// pattern evaluator's value stack and the texture filters next to both
// BSDFs, at two waves per SIMD (218-243 VGPRs without the fiber BSDF, so
// no smaller variant; a three-wave cap spills 140 VGPRs).
template <bool TR, bool FILM, bool FIXED>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(2))) void shade_pattern_kernel(
    PtSceneView S, PathBuffers P, PtParams prm, const uint32_t* __restrict__ q, uint32_t* __restrict__ qnext,
    NrcPathBuffers N) {
  shade_pass<false, TR, FILM, FIXED, true, true>(S, P, prm, q, qnext, N);
}
// The shade kernel for the pass's cache, film, transparency and hair, with
// render.rs's fixed origin push (FIXED) or error-bounded origins (caches
// are never attached to scenes with hair).
template <bool FIXED>
void launch_shade(const PtSceneView& S, const PathBuffers& P, const PtParams& prm, const uint32_t* qshade,
                  uint32_t* qnext, const NrcPathBuffers& N, uint32_t g, hipStream_t st) {
  const dim3 G(g), B(kBlock);
  if (S.patterns) {
    if (P.ld && S.transparent)
      hipLaunchKernelGGL((shade_pattern_kernel<true, true, FIXED>), G, B, 0, st, S, P, prm, qshade, qnext, N);
    else if (P.ld)
      hipLaunchKernelGGL((shade_pattern_kernel<false, true, FIXED>), G, B, 0, st, S, P, prm, qshade, qnext, N);
    else if (S.transparent)
      hipLaunchKernelGGL((shade_pattern_kernel<true, false, FIXED>), G, B, 0, st, S, P, prm, qshade, qnext, N);
    else
      hipLaunchKernelGGL((shade_pattern_kernel<false, false, FIXED>), G, B, 0, st, S, P, prm, qshade, qnext, N);
  } else if (S.hair) {
    if (P.ld && S.transparent)
      hipLaunchKernelGGL((shade_hair_kernel<true, true, FIXED>), G, B, 0, st, S, P, prm, qshade, qnext, N);
    else if (P.ld)
      hipLaunchKernelGGL((shade_hair_kernel<false, true, FIXED>), G, B, 0, st, S, P, prm, qshade, qnext, N);
    else if (S.transparent)
      hipLaunchKernelGGL((shade_hair_kernel<true, false, FIXED>), G, B, 0, st, S, P, prm, qshade, qnext, N);
    else
      hipLaunchKernelGGL((shade_hair_kernel<false, false, FIXED>), G, B, 0, st, S, P, prm, qshade, qnext, N);
  } else if (N.q) {
    hipLaunchKernelGGL((shade_kernel<true, false, false, FIXED>), G, B, 0, st, S, P, prm, qshade, qnext, N);
  } else if (P.ld && S.transparent) {
    hipLaunchKernelGGL((shade_kernel<false, true, true, FIXED>), G, B, 0, st, S, P, prm, qshade, qnext, N);
  } else if (P.ld) {
    hipLaunchKernelGGL((shade_kernel<false, false, true, FIXED>), G, B, 0, st, S, P, prm, qshade, qnext, N);
  } else if (S.transparent) {
    hipLaunchKernelGGL((shade_kernel<false, true, false, FIXED>), G, B, 0, st, S, P, prm, qshade, qnext, N);
  } else {
    hipLaunchKernelGGL((shade_kernel<false, false, false, FIXED>), G, B, 0, st, S, P, prm, qshade, qnext, N);
  }
}

}  // namespace

hipError_t pt_launch_shade(const PtSceneView& S, const PathBuffers& P, const PtParams& prm, const uint32_t* qshade,
                           uint32_t* qnext, const NrcPathBuffers& N, uint32_t g, hipStream_t st) {
  if (S.ray_offset > 0.f)
    launch_shade<true>(S, P, prm, qshade, qnext, N, g, st);
  else
    launch_shade<false>(S, P, prm, qshade, qnext, N, g, st);
  return hipGetLastError();
}

}  // namespace rrhip
