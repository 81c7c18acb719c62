// Shading kernels of the wavefront path integrator and their launch for one
// rule of ray origins (pt_shade_bounded.hip, pt_shade_fixed.hip: one each, so
// that they compile in parallel).
#pragma once
#include <hip/hip_runtime.h>

#include "pt_wave.h"

namespace rrhip {
namespace {

using namespace pt;

// Waves per SIMD: three without media (145 to 160 registers). The media
// code (distance sampling, ratio tracking, equiangular connections) takes
// the surface lobes to 218-228 registers, and under a three-wave cap it
// spilled 96 to 168 B per lane to scratch in every scene; scenes without
// media therefore have kernels of their own, the others run two waves
// without spills (200 x 200 cloud room, 16 samples: 4.98 -> 4.48 ms of
// device time a frame; 256 x 256 box room: 1.19 -> 1.08).
template <bool NRC, bool TR, bool MEDIA, bool FILM = false, bool FIXED = false>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(MEDIA ? 2 : 3))) void shade_kernel(
    PtSceneView S, PathBuffers P, PtParams prm, const uint32_t* __restrict__ q, uint32_t* __restrict__ qnext,
    NrcPathBuffers N) {
  shade_pass<NRC, TR, MEDIA, FILM, FIXED, false>(S, P, prm, q, qnext, N);
}

// Scenes with hair fibers: the fiber BSDF's state next to the surface
// lobes' (166 registers without media, 222-232 with).
template <bool TR, bool MEDIA, bool FILM, bool FIXED>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(MEDIA ? 2 : 3))) void shade_hair_kernel(
    PtSceneView S, PathBuffers P, PtParams prm, const uint32_t* __restrict__ q, uint32_t* __restrict__ qnext,
    NrcPathBuffers N) {
  shade_pass<false, TR, MEDIA, FILM, FIXED, true>(S, P, prm, q, qnext, N);
}

// Scenes with pattern-bound materials (and hair fibers, if any): the
// pattern evaluator's value stack and the texture filters next to both
// BSDFs, at two waves per SIMD (212-226 registers without media).
template <bool TR, bool MEDIA, bool FILM, bool FIXED>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(2))) void shade_pattern_kernel(
    PtSceneView S, PathBuffers P, PtParams prm, const uint32_t* __restrict__ q, uint32_t* __restrict__ qnext,
    NrcPathBuffers N) {
  shade_pass<false, TR, MEDIA, FILM, FIXED, true, true>(S, P, prm, q, qnext, N);
}

// The shade kernel for the pass's cache, film and origin rule (FIXED:
// render.rs's fixed push, else error-bounded origins; caches are never
// attached to scenes with hair) and the scene's class: transparent scenes
// keep the media code, others carry it when every ray travels in an
// atmosphere.
template <bool TR, bool MEDIA, bool FILM, bool FIXED>
void launch_shade_class(const PtSceneView& S, const PathBuffers& P, const PtParams& prm, const uint32_t* qshade,
                        uint32_t* qnext, const NrcPathBuffers& N, uint32_t g, hipStream_t st) {
  const dim3 G(g), B(kBlock);
  if (S.patterns)
    hipLaunchKernelGGL((shade_pattern_kernel<TR, MEDIA, FILM, FIXED>), G, B, 0, st, S, P, prm, qshade, qnext, N);
  else if (S.hair)
    hipLaunchKernelGGL((shade_hair_kernel<TR, MEDIA, FILM, FIXED>), G, B, 0, st, S, P, prm, qshade, qnext, N);
  else
    hipLaunchKernelGGL((shade_kernel<false, TR, MEDIA, FILM, FIXED>), G, B, 0, st, S, P, prm, qshade, qnext, N);
}

template <bool FILM, bool FIXED>
void launch_shade_film(const PtSceneView& S, const PathBuffers& P, const PtParams& prm, const uint32_t* qshade,
                       uint32_t* qnext, const NrcPathBuffers& N, uint32_t g, hipStream_t st) {
  if (S.transparent)
    launch_shade_class<true, true, FILM, FIXED>(S, P, prm, qshade, qnext, N, g, st);
  else if (S.atmosphere >= 0)
    launch_shade_class<false, true, FILM, FIXED>(S, P, prm, qshade, qnext, N, g, st);
  else
    launch_shade_class<false, false, FILM, FIXED>(S, P, prm, qshade, qnext, N, g, st);
}

// The shading kernel of one bounce: the radiance cache's (caches are never
// attached to scenes with hair, patterns or media), or the film mode's.
template <bool FIXED>
hipError_t launch_shade(const PtSceneView& S, const PathBuffers& P, const PtParams& prm, const uint32_t* qshade,
                        uint32_t* qnext, const NrcPathBuffers& N, uint32_t g, hipStream_t st) {
  if (N.q && !S.patterns && !S.hair)
    hipLaunchKernelGGL((shade_kernel<true, false, false, false, FIXED>), dim3(g), dim3(kBlock), 0, st, S, P, prm,
                       qshade, qnext, N);
  else if (P.ld)
    launch_shade_film<true, FIXED>(S, P, prm, qshade, qnext, N, g, st);
  else
    launch_shade_film<false, FIXED>(S, P, prm, qshade, qnext, N, g, st);
  return hipGetLastError();
}

}  // namespace
}  // namespace rrhip
