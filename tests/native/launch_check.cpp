// Launches that must be refused before anything reaches a device, for
// test_launch_rules.py.
#include <hip/hip_runtime.h>

#include "pt_kernels.h"

using namespace rrhip;

extern "C" {

// The status of a trace launch over an empty scene; 0 if it was let through
// to the launch (which fails without a device).
int check_trace(int transparent, int profiled, int queue, int work) {
  PtSceneView S{};
  PathBuffers P{};
  static uint32_t q[1];
  static unsigned long long prof[8];
  S.transparent = (uint32_t)transparent;
  P.prof = profiled ? prof : nullptr;
  const hipError_t e = pt_launch_trace(S, P, queue ? q : nullptr, 1, (TraceWork)work, nullptr);
  return e == hipErrorInvalidValue ? (int)e : 0;
}

}  // extern "C"
