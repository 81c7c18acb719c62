// The ends of a pass's paths in one launch: once few paths are left, every
// lane carries one through its remaining bounces by itself.
#include <hip/hip_runtime.h>

#include "pt_wave.h"

namespace rrhip {
namespace {

using namespace pt;

// Continues the live paths of round P.round, whose closest hits are known,
// to their ends when there are at most `limit` of them: shading, the shadow
// record evaluated in place (record index = path slot), the next closest
// hit, and again.
//
// A bounce round takes two launches and lasts at least as long as its
// slowest path, and with few paths left that is nearly all of it: the 48
// last of a cloud room's 64 rounds took 25 to 40 us each for less than a
// tenth of the paths. Here a pass waits once for its longest path instead of
// once a round. Two waves per SIMD, so that shading does not spill; a wave
// refills its idle lanes from its run of the queue. 200 x 200 cloud room, 16
// samples, 64 bounces: 3.90 -> 3.10 ms of device time a frame (300 x 290:
// 5.87 -> 4.97, 150 x 140 with 3 samples: 1.98 -> 1.39); 960 x 540 instanced
// field through the radiance cache, 4 samples, 12 bounces: 8.45 -> 7.91.
template <bool NRC, bool MEDIA, bool FILM>
__global__ __launch_bounds__(kTraceBlock) __attribute__((amdgpu_waves_per_eu(2))) void tail_kernel(
    PtSceneView S, PathBuffers P, PtParams prm, const uint32_t* __restrict__ q, NrcPathBuffers N, uint32_t limit) {
  __shared__ uint32_t s_stack[kTraceStack * kTraceBlock];
  uint32_t* stk = s_stack + threadIdx.x;
  const uint32_t n = P.live();
  if (n == 0 || n > limit) return;
  // every resident wave takes an equal run of the queue
  const uint32_t waves = gridDim.x * (kTraceBlock / 64);
  const uint32_t wave = __builtin_amdgcn_readfirstlane((blockIdx.x * kTraceBlock + threadIdx.x) >> 6);
  const uint32_t share = (n + waves - 1) / waves;
  uint32_t next = min(n, wave * share);
  const uint32_t end = min(n, next + share);
  const auto rank = [](uint64_t m) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
  };
  unsigned long long ext = 0, shd = 0;
  uint32_t slot = 0;
  bool have = false;
  for (;;) {
    const uint64_t idle = __ballot(!have);
    if (idle && next < end) {
      const uint32_t i = next + rank(idle);
      if (!have && i < end) {
        slot = q[i];
        have = true;
      }
      next += __popcll(idle);
    }
    if (!__ballot(have)) break;
    bool cont = false, shadow = false, shadow2 = false, query = false;
    ShadowOut so, se;
    NrcQuery nq;
    V3 qbeta;
    if (have)
      shade_one<NRC, false, FILM, false, false, false, MEDIA>(S, P, prm, N, slot, cont, shadow, shadow2, se, query, so, nq,
                                                          qbeta);
    if constexpr (NRC) {
      const uint64_t m = __ballot(query);
      if (m) {
        uint32_t base = 0;
        if (rank(m) == 0 && query) base = atomicAdd(&N.counts[0], (uint32_t)__popcll(m));
        base = __shfl(base, (int)(__ffsll((unsigned long long)m) - 1));
        if (query) {
          const uint32_t i = base + rank(m);
          N.q[i] = nq;
          N.q_slot[i] = slot;
          N.q_beta[i] = make_float4(qbeta.x, qbeta.y, qbeta.z, 0.f);
        }
      }
    }
    if (shadow || shadow2) {
      put_shadow<false, FILM>(P, slot, slot, shadow, so, shadow2, se);
      shadow_one_t<false, false, 0>(S, P, slot, stk);
      shd++;
    }
    have = cont;
    if (cont) {
      extend_one<false, 0>(S, P, slot, stk);
      ext++;
    }
  }
  for (int off = 32; off > 0; off >>= 1) {
    ext += __shfl_xor(ext, off);
    shd += __shfl_xor(shd, off);
  }
  if ((threadIdx.x & 63u) == 0) {
    if (ext) atomicAdd(P.stats + 0, ext);
    if (shd) atomicAdd(P.stats + 1, shd);
  }
}

using TailFn = void (*)(PtSceneView, PathBuffers, PtParams, const uint32_t*, NrcPathBuffers, uint32_t);

// The kernel of a pass's scene class; null where the rounds run to the end.
// Media and the cache leave most rounds few paths. Opaque scenes without
// them keep more than 65,536 to their last bounce at the sizes where a frame
// takes long: no gain on the 540p field and the box room, and finishing
// 196,608 paths of a fur ball here, at two waves per SIMD, was slower than
// its rounds (14.4 against 12.9 ms).
TailFn tail_fn(const PtSceneView& S, const PathBuffers& P, const NrcPathBuffers& N) {
  if (P.prof || S.transparent || S.patterns || S.motion || S.num_quadrics || S.ray_offset > 0.f || S.curves || S.hair)
    return nullptr;
  const bool media = S.atmosphere >= 0;
  if (N.q) return media || P.ld ? nullptr : (TailFn)tail_kernel<true, false, false>;
  if (!media) return nullptr;
  return P.ld ? (TailFn)tail_kernel<false, true, true> : (TailFn)tail_kernel<false, true, false>;
}

}  // namespace

// 65,536 paths are half of the lanes that the card holds of this kernel
// and what its rounds no longer fill (131,072: cloud room 3.10 -> 3.18 ms,
// cache field 7.91 -> 7.75). Asking in more rounds (2, 6, or each from 4 to
// 8) or ending at round 32 instead of 16 changed no case by more than 2 %.
// After round 16 any number ends here, which saves the launches of up to 47
// rounds: also where a cloud ten times as dense without absorption keeps
// most of 2.6 million paths alive, that costs 1.5 % (47.1 -> 47.9 ms).
uint32_t pt_tail_limit(const PtSceneView& S, const PathBuffers& P, const NrcPathBuffers& N) {
  if (!tail_fn(S, P, N)) return 0;
  if (P.round == 4 || P.round == 8 || P.round == 12) return 65536;
  return P.round == 16 ? 0xFFFFFFFFu : 0;
}

hipError_t pt_launch_tail(const PtSceneView& S, const PathBuffers& P, const PtParams& prm, const uint32_t* q,
                          const NrcPathBuffers& N, uint32_t limit, hipStream_t st) {
  hipLaunchKernelGGL(tail_fn(S, P, N), dim3(1024), dim3(kTraceBlock), 0, st, S, P, prm, q, N, limit);
  return hipGetLastError();
}

}  // namespace rrhip
