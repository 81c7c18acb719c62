// Batched jobs in one persistent launch (render.rs renders scenes one by
// one).
#include <hip/hip_runtime.h>

#include "pt_wave.h"

namespace rrhip {
namespace {

using namespace pt;

constexpr uint32_t kOpenChunks = 64;  // chunks a wave can have open at once

// ---- batched jobs in one persistent launch ---------------------------------------
// Every lane owns one path slot. A wave pulls chunks of a job — as many whole
// pixels as make up at most 64 samples — from a device counter until the
// chunks run out, and deals their samples to its lanes as these fall idle;
// chunks are numbered job by job (pix_begin) in the order the host chose
// (shortest job first). A path runs through the same device functions the
// wavefront kernels call (camera ray, closest hit, shading, shadow records
// evaluated in place). Its radiance waits in the wave's part of `samples`
// until the chunk's last path is done: then a lane per pixel adds the
// samples in order into the pixel's accumulator row. The last pixels of a
// job record the device clock, so per-job completion is measured inside the
// one launch. There are no barriers: a wave exits when the counter passes
// the last chunk and its paths are done.
//
// Bound by latency at two waves per SIMD (the registers of media shading)
// and 25 lanes per vector instruction. With a pixel and all its samples per
// lane, the lanes that drew the last pixels of the longest job ran up to 16
// paths one after another while the others had ended, and the lanes of a
// wave drifted apart into different jobs: 16 rooms of up to 256 x 256
// pixels and 16 samples 15.5 -> 11.7 ms. Slower: the job's scene in scalar
// registers, one job of the wave after another (16.8 ms, with or without
// shading code of its own for jobs without media).

// One bounce of the path in slot `slot` (closest hit, shading, its shadow
// record evaluated in place); returns whether the path continues and
// counts rays and shadow records. TR: the job is transparent (its own
// scene's flag, as its session shades it); MOTION / QUAD: some job of the
// batch moves / holds quadrics (the kernel is instantiated for the
// batch's union of them; static and quadric-free scenes take the same
// paths through those templates).
template <bool TR, bool MOTION, bool QUAD>
__device__ __forceinline__ bool persist_bounce(const PtJob& J, const PathBuffers& P, uint32_t slot, uint32_t* stk,
                                               unsigned long long& ext, unsigned long long& shd) {
  const NrcPathBuffers N{};
  extend_one<MOTION, QUAD ? 3 : 0>(J.S, P, slot, stk);
  ext++;
  bool cont = false, shadow = false, shadow2 = false, query = false;
  ShadowOut so, se;
  NrcQuery nq;
  V3 qbeta;
  shade_one<false, TR>(J.S, P, J.prm, N, slot, cont, shadow, shadow2, se, query, so, nq, qbeta);
  if (shadow || shadow2) {
    put_shadow<TR>(P, slot, slot, shadow, so, shadow2, se);
    shadow_one_t<TR, MOTION, QUAD ? 3 : 0>(J.S, P, slot, stk);
    shd++;
  }
  return cont;
}

// The sample as resolve_one adds it (firefly clamp on luminance): l, and
// its luminance returned.
__device__ __forceinline__ double clamped_sample(const float4& l4, float firefly_clamp, double l[3]) {
  l[0] = l4.x;
  l[1] = l4.y;
  l[2] = l4.z;
  double lm = 0.2126 * l[0] + 0.7152 * l[1] + 0.0722 * l[2];
  if (firefly_clamp > 0.f && lm > (double)firefly_clamp) {
    const double sc = (double)firefly_clamp / lm;
    l[0] *= sc;
    l[1] *= sc;
    l[2] *= sc;
    lm = 0.2126 * l[0] + 0.7152 * l[1] + 0.0722 * l[2];
  }
  return lm;
}

// Adds samples [0, n) of a pixel, in order, to its accumulator row.
__device__ __forceinline__ void add_samples(double* a, const float4* L, uint32_t n, float firefly_clamp) {
  double sum[3] = {0, 0, 0}, sq[3] = {0, 0, 0}, ql = 0.0;
  for (uint32_t k = 0; k < n; k++) {
    double l[3];
    const double lm = clamped_sample(L[k], firefly_clamp, l);
    for (int c = 0; c < 3; c++) {
      sum[c] += l[c];
      sq[c] += l[c] * l[c];
    }
    ql += lm * lm;
  }
  for (int c = 0; c < 3; c++) {
    a[c] += sum[c];
    a[3 + c] += sq[c];
  }
  a[6] += (double)n;
  a[7] += ql;
}

// A wave runs one flat loop of bounces: lanes whose path ended take the next
// samples of the wave's chunk in the same iteration, so no lane waits for
// the others' paths. Up to 64 chunks are open at once (each but the one that
// is being dealt has a path in some lane); `cfree` marks the wave's free
// parts of `samples`. Jobs of more than kPtChunkSamples samples per pixel have
// no place there: a lane runs all samples of such a pixel and adds them to
// its row one by one.
template <bool TR, bool MOTION, bool QUAD>
__global__ __launch_bounds__(kTraceBlock) __attribute__((amdgpu_waves_per_eu(2))) void batch_persistent_kernel(
    const PtJob* __restrict__ jobs, uint32_t nj, PathBuffers P, uint32_t total_items, uint32_t* __restrict__ next_item,
    uint32_t* __restrict__ job_left, unsigned long long* __restrict__ job_clock, float4* samples) {
  __shared__ uint32_t s_stack[kTraceStack * kTraceBlock];
  uint32_t* stk = s_stack + threadIdx.x;
  const uint32_t slot = blockIdx.x * blockDim.x + threadIdx.x, lane = threadIdx.x & 63u;
  if (threadIdx.x == 0) atomicMin(job_clock + nj, (unsigned long long)wall_clock64());
  float4* const wave_samples =
      samples + (size_t)__builtin_amdgcn_readfirstlane(slot >> 6) * (kOpenChunks * kPtChunkSamples);
  unsigned long long ext = 0, shd = 0;
  // the chunk being dealt: its job, first pixel, samples (or pixels) dealt
  // and in all, part of `samples`
  uint32_t cj = 0, cpix = 0, cnext = 0, cunits = 0, cpart = 0;
  uint64_t cfree = ~0ull;
  bool drained = false;
  // the lane's path
  uint32_t j = 0, pixel = 0, first = 0, k = 0, part = kOpenChunks, unit = 0, b = 0, rounds = 0;
  bool have = false, start = false;
  for (;;) {
    for (uint64_t idle = __ballot(!have); idle && !drained; idle = __ballot(!have)) {
      if (cnext == cunits) {
        uint32_t item = 0;
        if (lane == 0) item = atomicAdd(next_item, 1u);
        item = __builtin_amdgcn_readfirstlane(item);
        if (item >= total_items) {
          drained = true;
          break;
        }
        cj = __builtin_amdgcn_readfirstlane(find_job<true>(jobs, nj, item));
        const PtJob& J = jobs[cj];
        cpix = (item - J.pix_begin) * J.chunk_pix;
        const uint32_t np = min(J.chunk_pix, J.prm.npix - cpix);
        cunits = J.prm.spp_pass > kPtChunkSamples ? np : np * J.prm.spp_pass;
        cnext = 0;
        cpart = (uint32_t)__ffsll((unsigned long long)cfree) - 1u;
        cfree &= ~(1ull << cpart);
      }
      const uint32_t u = cnext + __builtin_amdgcn_mbcnt_hi((uint32_t)(idle >> 32),
                                                           __builtin_amdgcn_mbcnt_lo((uint32_t)idle, 0u));
      if (!have && u < cunits) {
        const uint32_t spp = jobs[cj].prm.spp_pass;
        const bool whole = spp > kPtChunkSamples;
        j = cj;
        first = cpix;
        part = cpart;
        unit = u;
        pixel = cpix + (whole ? u : u / spp);
        k = whole ? 0u : u % spp;
        have = start = true;
      }
      cnext = min(cunits, cnext + (uint32_t)__popcll(idle));
    }
    if (!__ballot(have)) break;
    bool ended = false;
    if (have) {
      const PtJob& J = jobs[j];
      if (start) {
        init_path(J.S, P, slot, pixel, J.prm.sample0 + k, kFlagFromCamera);
        rounds = J.prm.max_depth + (TR && J.S.transparent ? kPtMaxSkips : 0);
        b = 0;
        start = false;
      }
      const bool cont = TR && J.S.transparent ? persist_bounce<true, MOTION, QUAD>(J, P, slot, stk, ext, shd)
                                              : persist_bounce<false, MOTION, QUAD>(J, P, slot, stk, ext, shd);
      if (!cont || ++b >= rounds) {
        if (J.prm.spp_pass > kPtChunkSamples) {
          add_samples(J.accum + 8 * (size_t)pixel, P.L + slot, 1, J.prm.firefly_clamp);
          start = true;
          ended = ++k == J.prm.spp_pass;
        } else {
          wave_samples[part * kPtChunkSamples + unit] = P.L[slot];
          ended = true;
        }
        if (ended) have = false;
      }
    }
    uint64_t done = __ballot(ended);
    if (!done) continue;
    __threadfence_block();  // the samples are the wave's own: its stores before its loads
    while (done) {
      const int l0 = __ffsll((unsigned long long)done) - 1;
      const uint32_t c = __builtin_amdgcn_readlane(part, l0);
      done &= ~__ballot(ended && part == c);
      if (__ballot(have && part == c) || (c == cpart && cnext < cunits)) continue;
      // the chunk's last path
      const uint32_t jj = __builtin_amdgcn_readlane(j, l0), p0 = __builtin_amdgcn_readlane(first, l0);
      const PtJob& J = jobs[jj];
      const uint32_t np = min(J.chunk_pix, J.prm.npix - p0), spp = J.prm.spp_pass;
      if (spp <= kPtChunkSamples && lane < np)
        add_samples(J.accum + 8 * (size_t)(p0 + lane), wave_samples + c * kPtChunkSamples + lane * spp, spp,
                    J.prm.firefly_clamp);
      cfree |= 1ull << c;
      if (lane == 0 && atomicSub(job_left + jj, np) == np) job_clock[jj] = wall_clock64();
    }
  }
  // rays traced (per wave, one atomic); every lane of the wave has left the
  // loop here
  for (int off = 32; off > 0; off >>= 1) {
    ext += __shfl_xor(ext, off);
    shd += __shfl_xor(shd, off);
  }
  if ((threadIdx.x & 63u) == 0) {
    atomicAdd(P.stats + 0, ext);
    atomicAdd(P.stats + 1, shd);
  }
}

// The persistent kernel of a batch's flags (flags bit 0 transparent, 1
// motion, 2 quadrics).
using PersistFn = void (*)(const PtJob*, uint32_t, PathBuffers, uint32_t, uint32_t*, uint32_t*, unsigned long long*,
                           float4*);
PersistFn persist_fn(uint32_t flags) {
  switch (flags & 7u) {
    case 0: return batch_persistent_kernel<false, false, false>;
    case 1: return batch_persistent_kernel<true, false, false>;
    case 2: return batch_persistent_kernel<false, true, false>;
    case 3: return batch_persistent_kernel<true, true, false>;
    case 4: return batch_persistent_kernel<false, false, true>;
    case 5: return batch_persistent_kernel<true, false, true>;
    case 6: return batch_persistent_kernel<false, true, true>;
    default: return batch_persistent_kernel<true, true, true>;
  }
}
}  // namespace

hipError_t pt_launch_batch_persistent(const PtJob* jobs, uint32_t nj, const PathBuffers& P, uint32_t total_items,
                                      uint32_t lanes, uint32_t flags, uint32_t* next_item, uint32_t* job_left,
                                      unsigned long long* job_clock, float4* samples, hipStream_t st) {
  hipLaunchKernelGGL(persist_fn(flags), dim3(lanes / kTraceBlock), dim3(kTraceBlock), 0, st, jobs, nj, P,
                     total_items, next_item, job_left, job_clock, samples);
  return hipGetLastError();
}

uint32_t pt_batch_persistent_lanes(uint32_t flags) {
  int dev = 0, cus = 0, per_cu = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 0;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, persist_fn(flags), kTraceBlock, 0) != hipSuccess)
    return 0;
  if (per_cu <= 0 || cus <= 0) return 0;
  return (uint32_t)(per_cu * cus) * kTraceBlock;
}

}  // namespace rrhip
