// Shading kernels with render.rs's fixed push of ray origins.
#include "pt_shade.h"

namespace rrhip {

hipError_t pt_launch_shade_fixed(const PtSceneView& S, const PathBuffers& P, const PtParams& prm,
                              const uint32_t* qshade, uint32_t* qnext, const NrcPathBuffers& N, uint32_t g,
                              hipStream_t st) {
  return launch_shade<true>(S, P, prm, qshade, qnext, N, g, st);
}

}  // namespace rrhip
