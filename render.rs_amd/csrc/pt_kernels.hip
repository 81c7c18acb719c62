// Wavefront path integrator kernels for gfx950.
//
// The CPU path's loop body (render.rs src/raytracer/pt/mod.rs:449-990:
// intersect -> miss/dome -> emission with MIS -> NEE through the light BVH
// -> BSDF continuation -> Russian roulette) is split into stages that run
// over queues of live paths, so a wave only ever holds paths at the same
// stage and dead paths drop out of the launch instead of idling lanes
// (render.rs's own wavefront scheduler, kernel_wf.metal:1-20, does the
// same with one extend and one shade kernel). Shadow rays are queued for
// any-hit queries: in opaque scenes in the launch of the next round's closest
// hits, in transparent ones and while profiling in a launch of their own. In
// scenes with an atmosphere and in passes through the radiance cache the last
// paths end in a tail launch.
//
// Queue appends take one atomic per block. Results do not depend on queue
// order: every path owns its state, and pixels are accumulated by the
// resolve kernel in sample order, so renders are bit-reproducible.
//
// Here: camera rays, resolve and film kernels, the batched jobs' passes, the
// queue sort, and the launches of a bounce round. The trace, shade, tail and
// persistent batch kernels have files of their own.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "pt_wave.h"

namespace rrhip {
namespace {

using namespace pt;

// The first `count` u32 draws of the per-(pixel, sample) streams, seeded
// exactly as init_path seeds a camera path: out[i * count + k].
__global__ __launch_bounds__(kBlock) void pcg32_draws_kernel(const uint64_t* __restrict__ pixel,
                                                            const uint64_t* __restrict__ sample, uint32_t n,
                                                            uint32_t count, uint32_t* __restrict__ out) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  Pcg32 rng = Pcg32::for_pixel_sample(pixel[i], sample[i]);
  for (uint32_t k = 0; k < count; k++) out[(size_t)i * count + k] = rng.next_u32();
}

// The round words of a pass that starts with n paths.
__device__ __forceinline__ void start_rounds(const PathBuffers& P, uint32_t n) {
  for (uint32_t i = threadIdx.x; i < kRoundWords; i += blockDim.x) P.rounds[i] = i == 0 ? n : 0;
}

// sample0_dev (when set) supplies the pass's first sample index from device
// memory, so a captured pass graph can be replayed for any sample range.
__global__ __launch_bounds__(kBlock) void raygen_kernel(PtSceneView S, PathBuffers P, PtParams prm, uint32_t total,
                                                       NrcPathBuffers N, const uint64_t* __restrict__ sample0_dev) {
  if (sample0_dev) prm.sample0 = *sample0_dev;
  const uint32_t all = total + N.ntrain;
  if (blockIdx.x == 0) start_rounds(P, all);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    // N.counts[1] (training samples of the previous pass) is left alone: the
    // previous pass's optimiser steps may still be reading it, and this
    // pass's scan overwrites it before its own steps.
    if (N.counts) N.counts[0] = 0;
  }
  const uint32_t stride = gridDim.x * blockDim.x;
  for (uint32_t slot = blockIdx.x * blockDim.x + threadIdx.x; slot < all; slot += stride) {
    uint32_t pixel, flags = kFlagFromCamera;
    uint64_t sample;
    if (slot < total) {
      pixel = slot % prm.npix;
      sample = prm.sample0 + slot / prm.npix;
      if (prm.live) pixel = prm.live[pixel];
    } else {
      // Training path i of this pass: a hashed pixel and a PCG32 stream of
      // its own (top bit set: never a rendering sample index).
      const uint32_t i = slot - total;
      const uint64_t tag = ((prm.sample0 << 22) | i) & 0x7FFFFFFFFFFFFFFFull;
      pixel = (uint32_t)(Pcg32::mix(tag ^ 0x6e72637472616e69ull) % prm.npix);
      if (prm.live) pixel = prm.live[pixel];
      sample = 0x8000000000000000ull | tag;
      flags |= kFlagTrain;
      N.tn[i] = 0;
    }
    init_path(S, P, slot, pixel, sample, flags);
  }
}

// Adds the rays of rounds [0, P.round) to the session's totals.
__device__ __forceinline__ void add_ray_totals(const PathBuffers& P) {
  for (uint32_t i = threadIdx.x; i <= P.round; i += blockDim.x) {
    const unsigned long long w = P.rounds[i];
    if (i < P.round && (uint32_t)w) atomicAdd(P.stats + 0, (unsigned long long)(uint32_t)w);
    if (w >> 32) atomicAdd(P.stats + 1, w >> 32);
  }
}

__global__ __launch_bounds__(kBlock) void resolve_kernel(PathBuffers P, PtParams prm, double* __restrict__ accum) {
  if (blockIdx.x == 0) add_ray_totals(P);
  const uint32_t stride = gridDim.x * blockDim.x;
  for (uint32_t c = blockIdx.x * blockDim.x + threadIdx.x; c < prm.npix; c += stride) resolve_one(P, prm, accum, c, 0);
}

// Film accumulators of column col's pass samples, in sample order
// (pt/mod.rs:200-221): the diffuse split with the sample's firefly scale,
// albedo and normal sums, the depth sum and count over samples with a
// first real hit, and the id vote (kFilmIds slots of id and count, then
// the count of samples whose id found no slot).
__device__ __forceinline__ void resolve_film_one(const PathBuffers& P, const PtParams& prm, double* film,
                                                 uint32_t col) {
  const uint32_t px = prm.live ? prm.live[col] : col;
  double* a = film + (size_t)kFilmStride * px;
  double ds[3] = {0, 0, 0}, al[3] = {0, 0, 0}, nm[3] = {0, 0, 0}, dep = 0.0, hits = 0.0, over = 0.0;
  uint32_t ids[kFilmIds], cnt[kFilmIds];
#pragma unroll
  for (int j = 0; j < (int)kFilmIds; j++) {
    ids[j] = (uint32_t)a[11 + j];
    cnt[j] = (uint32_t)a[11 + kFilmIds + j];
  }
  for (uint32_t k = 0; k < prm.spp_pass; k++) {
    const size_t slot = (size_t)k * prm.npix + col;
    const float4 l4 = P.L[slot], d4 = P.ld[slot], x0 = P.aux0[slot], x1 = P.aux1[slot];
    const uint32_t id = P.aux_id[slot];
    double sc = 1.0;
    const double lm = 0.2126 * (double)l4.x + 0.7152 * (double)l4.y + 0.0722 * (double)l4.z;
    if (prm.firefly_clamp > 0.f && lm > (double)prm.firefly_clamp) sc = (double)prm.firefly_clamp / lm;
    ds[0] += (double)d4.x * sc;
    ds[1] += (double)d4.y * sc;
    ds[2] += (double)d4.z * sc;
    al[0] += x0.x;
    al[1] += x0.y;
    al[2] += x0.z;
    nm[0] += x1.x;
    nm[1] += x1.y;
    nm[2] += x1.z;
    if (x0.w > 0.f) {
      dep += x0.w;
      hits += 1.0;
    }
    bool placed = false;
#pragma unroll
    for (int j = 0; j < (int)kFilmIds; j++) {
      if (!placed && cnt[j] != 0 && ids[j] == id) {
        cnt[j]++;
        placed = true;
      }
    }
#pragma unroll
    for (int j = 0; j < (int)kFilmIds; j++) {
      if (!placed && cnt[j] == 0) {
        ids[j] = id;
        cnt[j] = 1;
        placed = true;
      }
    }
    if (!placed) over += 1.0;
  }
  for (int c = 0; c < 3; c++) {
    a[c] += ds[c];
    a[3 + c] += al[c];
    a[6 + c] += nm[c];
  }
  a[9] += dep;
  a[10] += hits;
#pragma unroll
  for (int j = 0; j < (int)kFilmIds; j++) {
    a[11 + j] = (double)ids[j];
    a[11 + kFilmIds + j] = (double)cnt[j];
  }
  a[11 + 2 * kFilmIds] += over;
}

__global__ __launch_bounds__(kBlock) void resolve_film_kernel(PathBuffers P, PtParams prm, double* __restrict__ film) {
  const uint32_t stride = gridDim.x * blockDim.x;
  for (uint32_t c = blockIdx.x * blockDim.x + threadIdx.x; c < prm.npix; c += stride) resolve_film_one(P, prm, film, c);
}

// The film's channels of one pixel (pt/mod.rs:223-274): sample means;
// specular = max(beauty - diffuse, 0); depth over the samples with a first
// real hit; the most voted id (the first of equal counts) and its share of
// the samples. Bound by memory (64 + 160 B read and 144 B written a pixel);
// on the host this loop and the copies of both accumulators into fresh
// vectors took most of a 640 x 360 film's time, 224 B a pixel over the bus
// instead of 144: the frame of 16 spp with its read-back takes 7.9 ms, 18.9
// with the host loop.
__global__ __launch_bounds__(kBlock) void film_image_kernel(const double* __restrict__ accum,
                                                           const double* __restrict__ film, uint32_t npix,
                                                           double* __restrict__ out) {
  const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= npix) return;
  const double* a = accum + 8 * (size_t)p;
  const double* f = film + (size_t)kFilmStride * p;
  double* o = out + (size_t)kFilmChannels * p;
  const double n = a[6] > 0.0 ? a[6] : 1.0;
  for (int c = 0; c < 3; c++) {
    const double beauty = a[c] / n, diffuse = f[c] / n, rest = beauty - diffuse;
    o[c] = beauty;
    o[3 + c] = diffuse;
    o[6 + c] = rest < 0.0 ? 0.0 : rest;
    o[9 + c] = f[3 + c] / n;
    o[12 + c] = f[6 + c] / n;
  }
  o[15] = f[10] > 0.0 ? f[9] / f[10] : 0.0;
  double best_id = 0.0, best_n = 0.0;
  for (uint32_t j = 0; j < kFilmIds; j++) {
    if (f[11 + kFilmIds + j] > best_n) {
      best_n = f[11 + kFilmIds + j];
      best_id = f[11 + j];
    }
  }
  o[16] = best_id;
  o[17] = best_n / n;
}

// ---- batched jobs: one set of launches over the path slots of many scenes ----

__global__ __launch_bounds__(kBlock) void raygen_batch_kernel(const PtJob* __restrict__ jobs, uint32_t nj, PathBuffers P,
                                                             uint32_t total) {
  if (blockIdx.x == 0) start_rounds(P, total);
  const uint32_t stride = gridDim.x * blockDim.x;
  for (uint32_t slot = blockIdx.x * blockDim.x + threadIdx.x; slot < total; slot += stride) {
    const uint32_t j = find_job<false>(jobs, nj, slot);
    const PtJob& J = jobs[j];
    const uint32_t local = slot - J.slot_begin;
    init_path(J.S, P, slot, local % J.prm.npix, J.prm.sample0 + local / J.prm.npix, kFlagFromCamera);
    P.job[slot] = j;
  }
}

template <bool QUAD>
__global__ __launch_bounds__(kTraceBlock) void extend_batch_kernel(const PtJob* __restrict__ jobs, PathBuffers P,
                                                                  const uint32_t* __restrict__ q) {
  __shared__ uint32_t s_stack[kTraceStack * kTraceBlock];
  uint32_t* stk = s_stack + threadIdx.x;
  const uint32_t n = P.live();
  const uint32_t stride = gridDim.x * blockDim.x;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const uint32_t slot = q[i];
    const PtSceneView& S = jobs[P.job[slot]].S;
    if (S.motion)
      extend_one<true, QUAD ? 3 : 0>(S, P, slot, stk);
    else
      extend_one<false, QUAD ? 3 : 0>(S, P, slot, stk);
  }
}

__global__ __launch_bounds__(kBlock) void shade_batch_kernel(const PtJob* __restrict__ jobs, PathBuffers P,
                                                            const uint32_t* __restrict__ q, uint32_t* __restrict__ qnext) {
  const uint32_t n = P.live();
  const uint32_t stride = gridDim.x * blockDim.x;
  const NrcPathBuffers N{};
  for (uint32_t base = blockIdx.x * blockDim.x; base < n; base += stride) {
    const uint32_t i = base + threadIdx.x;
    const bool act = i < n;
    bool cont = false, shadow = false, shadow2 = false, query = false;
    ShadowOut so, se;
    NrcQuery nq;
    V3 qbeta;
    uint32_t slot = 0;
    if (act) {
      slot = q[i];
      const PtJob& J = jobs[P.job[slot]];
      const bool fixed = J.S.ray_offset > 0.f;
      if (J.S.transparent && fixed)
        shade_one<false, true, false, true>(J.S, P, J.prm, N, slot, cont, shadow, shadow2, se, query, so, nq, qbeta);
      else if (J.S.transparent)
        shade_one<false, true>(J.S, P, J.prm, N, slot, cont, shadow, shadow2, se, query, so, nq, qbeta);
      else if (fixed)
        shade_one<false, false, false, true>(J.S, P, J.prm, N, slot, cont, shadow, shadow2, se, query, so, nq, qbeta);
      else
        shade_one<false, false>(J.S, P, J.prm, N, slot, cont, shadow, shadow2, se, query, so, nq, qbeta);
    }
    uint32_t nidx, sidx, qidx;
    block_append<false>(P.append(), nullptr, cont, shadow || shadow2, false, nidx, sidx, qidx);
    if (shadow || shadow2) {
      if (P.srng)
        put_shadow<true>(P, sidx, slot, shadow, so, shadow2, se);
      else
        put_shadow<false>(P, sidx, slot, shadow, so, shadow2, se);
    }
    if (cont) qnext[nidx] = slot;
  }
}

template <bool QUAD>
__global__ __launch_bounds__(kTraceBlock) void shadow_batch_kernel(const PtJob* __restrict__ jobs, PathBuffers P) {
  __shared__ uint32_t s_stack[kTraceStack * kTraceBlock];
  uint32_t* stk = s_stack + threadIdx.x;
  const uint32_t n = P.shadows();
  const uint32_t stride = gridDim.x * blockDim.x;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    shadow_one<QUAD>(jobs[P.job[P.sq[i]]].S, P, i, stk);
}

__global__ __launch_bounds__(kBlock) void resolve_batch_kernel(const PtJob* __restrict__ jobs, uint32_t nj, PathBuffers P,
                                                              uint32_t total_pix) {
  if (blockIdx.x == 0) add_ray_totals(P);
  const uint32_t stride = gridDim.x * blockDim.x;
  for (uint32_t g = blockIdx.x * blockDim.x + threadIdx.x; g < total_pix; g += stride) {
    const PtJob& J = jobs[find_job<true>(jobs, nj, g)];
    resolve_one(P, J.prm, J.accum, g - J.pix_begin, J.slot_begin);
  }
}

// ---- shading-class sort of the live queue (before shade) ------------------------
// Key: 0 = miss, else the hit material's sort_key (1 + active-lobe mask).
// Counting sort over fixed contiguous block ranges: per-block histograms,
// one scan over (class, block), then each block scatters its range.
constexpr uint32_t kSortKeys = 33;
constexpr uint32_t kSortBlocks = 512;

__device__ __forceinline__ uint32_t sort_key(const PtSceneView& S, const PathBuffers& P, uint32_t slot) {
  if (P.hit_n[slot].w < 0.f) return 0;
  return S.materials[P.hit_m[slot] & 0x7FFFFFFFu].sort_key;
}

__device__ __forceinline__ void block_range(uint32_t n, uint32_t& b0, uint32_t& b1) {
  const uint32_t chunk = (n + kSortBlocks - 1) / kSortBlocks;
  b0 = min(n, blockIdx.x * chunk);
  b1 = min(n, b0 + chunk);
}

__global__ __launch_bounds__(kBlock) void sort_count_kernel(PtSceneView S, PathBuffers P, const uint32_t* __restrict__ q) {
  __shared__ uint32_t h[kSortKeys];
  for (uint32_t i = threadIdx.x; i < kSortKeys; i += blockDim.x) h[i] = 0;
  __syncthreads();
  uint32_t b0, b1;
  block_range(P.live(), b0, b1);
  for (uint32_t i = b0 + threadIdx.x; i < b1; i += blockDim.x) atomicAdd(&h[sort_key(S, P, q[i])], 1u);
  __syncthreads();
  for (uint32_t k = threadIdx.x; k < kSortKeys; k += blockDim.x) P.sort_hist[k * kSortBlocks + blockIdx.x] = h[k];
}

// Exclusive scan of the (class, block) counts in place.
__global__ __launch_bounds__(1024) void sort_scan_kernel(PathBuffers P) {
  __shared__ uint32_t part[1024];
  constexpr uint32_t n = kSortKeys * kSortBlocks;
  const uint32_t t = threadIdx.x;
  const uint32_t chunk = (n + 1023) / 1024;
  const uint32_t b = t * chunk, e = min(n, b + chunk);
  uint32_t s = 0;
  for (uint32_t i = b; i < e; i++) s += P.sort_hist[i];
  part[t] = s;
  __syncthreads();
  for (uint32_t off = 1; off < 1024; off <<= 1) {
    const uint32_t v = t >= off ? part[t - off] : 0u;
    __syncthreads();
    part[t] += v;
    __syncthreads();
  }
  uint32_t run = part[t] - s;
  for (uint32_t i = b; i < e; i++) {
    const uint32_t c = P.sort_hist[i];
    P.sort_hist[i] = run;
    run += c;
  }
}

__global__ __launch_bounds__(kBlock) void sort_scatter_kernel(PtSceneView S, PathBuffers P, const uint32_t* __restrict__ q) {
  __shared__ uint32_t cur[kSortKeys];
  for (uint32_t k = threadIdx.x; k < kSortKeys; k += blockDim.x) cur[k] = P.sort_hist[k * kSortBlocks + blockIdx.x];
  __syncthreads();
  uint32_t b0, b1;
  block_range(P.live(), b0, b1);
  for (uint32_t i = b0 + threadIdx.x; i < b1; i += blockDim.x) {
    const uint32_t slot = q[i];
    P.qs[atomicAdd(&cur[sort_key(S, P, slot)], 1u)] = slot;
  }
}

}  // namespace

__global__ void set_u64_kernel(uint64_t* dst, uint64_t v) { *dst = v; }

hipError_t pt_launch_raygen(const PtSceneView& S, const PathBuffers& P, const PtParams& prm, uint32_t total,
                            const NrcPathBuffers& N, const uint64_t* sample0_dev, hipStream_t st) {
  hipLaunchKernelGGL(raygen_kernel, dim3(grid_for((uint64_t)total + N.ntrain)), dim3(kBlock), 0, st, S, P, prm, total,
                     N, sample0_dev);
  return hipGetLastError();
}

hipError_t pt_launch_set_u64(uint64_t* dst, uint64_t v, hipStream_t st) {
  hipLaunchKernelGGL(set_u64_kernel, dim3(1), dim3(1), 0, st, dst, v);
  return hipGetLastError();
}

// Trace launches have a block per 128 queue entries, as far as the capacity
// tells: blocks beyond the live paths end at once, and the dispatcher
// balances rays of very different length better than 4,096 striding blocks
// did (540p instanced field, 8 samples: 20.2 -> 18.6 ms of device time a
// frame).
static uint32_t trace_grid(uint64_t capacity) {
  const uint64_t b = (capacity + kTraceBlock - 1) / kTraceBlock;
  return (uint32_t)std::min<uint64_t>(65536, std::max<uint64_t>(1, b));
}

hipError_t pt_launch_bounce(const PtSceneView& S, PathBuffers P, const PtParams& prm, const uint32_t* q,
                            uint32_t* qnext, uint32_t capacity, const NrcPathBuffers& N, hipStream_t st,
                            const hipEvent_t* ev) {
  const uint32_t g = grid_for(capacity);
  // the counting kernels end with a few same-address atomics per wave, so
  // they keep to fewer, striding waves
  const uint32_t gt = P.prof ? grid_for(capacity, kTraceBlock) : trace_grid(capacity);
  const bool merged = !P.prof && !S.transparent;
  if (ev) (void)hipEventRecord(ev[0], st);
  hipError_t e = pt_launch_trace(S, P, q, gt, merged ? kTraceRound : kTraceExtend, st);
  if (e != hipSuccess) return e;
  if (ev) (void)hipEventRecord(ev[1], st);
  P.taken = pt_tail_limit(S, P, N);
  if (P.taken) {
    e = pt_launch_tail(S, P, prm, q, N, P.taken, st);
    if (e != hipSuccess || P.taken == 0xFFFFFFFFu) return e;
  }
  const uint32_t* qshade = q;
  if (P.qs) {  // group the queue by shading class so shade waves run one BSDF kind
    hipLaunchKernelGGL(sort_count_kernel, dim3(kSortBlocks), dim3(kBlock), 0, st, S, P, q);
    hipLaunchKernelGGL(sort_scan_kernel, dim3(1), dim3(1024), 0, st, P);
    hipLaunchKernelGGL(sort_scatter_kernel, dim3(kSortBlocks), dim3(kBlock), 0, st, S, P, q);
    qshade = P.qs;
  }
  e = S.ray_offset > 0.f ? pt_launch_shade_fixed(S, P, prm, qshade, qnext, N, g, st)
                         : pt_launch_shade_bounded(S, P, prm, qshade, qnext, N, g, st);
  if (e != hipSuccess) return e;
  if (ev) (void)hipEventRecord(ev[2], st);
  if (!merged) {
    PathBuffers Q = P;
    Q.round = P.round + 1;  // the records this round wrote
    e = pt_launch_trace(S, Q, nullptr, gt, kTraceShadow, st);
    if (e != hipSuccess) return e;
  }
  if (ev) (void)hipEventRecord(ev[3], st);
  return hipGetLastError();
}

hipError_t pt_launch_last_shadows(const PtSceneView& S, const PathBuffers& P, uint32_t capacity, hipStream_t st) {
  if (P.prof || S.transparent) return hipSuccess;
  return pt_launch_trace(S, P, nullptr, trace_grid(capacity), kTraceShadow, st);
}

hipError_t pt_launch_batch_pass(const PtJob* jobs, uint32_t nj, PathBuffers P, uint32_t total,
                                 uint32_t total_pix, uint32_t bounces, bool quadrics, hipStream_t st) {
  const uint32_t g = grid_for(total);
  const uint32_t gt = trace_grid(total);
  hipLaunchKernelGGL(raygen_batch_kernel, dim3(g), dim3(kBlock), 0, st, jobs, nj, P, total);
  for (uint32_t b = 0; b < bounces; b++) {
    P.round = b;
    const uint32_t* q = (b & 1) ? P.q1 : P.q0;
    uint32_t* qn = (b & 1) ? P.q0 : P.q1;
    if (quadrics)
      hipLaunchKernelGGL(extend_batch_kernel<true>, dim3(gt), dim3(kTraceBlock), 0, st, jobs, P, q);
    else
      hipLaunchKernelGGL(extend_batch_kernel<false>, dim3(gt), dim3(kTraceBlock), 0, st, jobs, P, q);
    hipLaunchKernelGGL(shade_batch_kernel, dim3(g), dim3(kBlock), 0, st, jobs, P, q, qn);
    P.round = b + 1;  // the records this round wrote
    if (quadrics)
      hipLaunchKernelGGL(shadow_batch_kernel<true>, dim3(gt), dim3(kTraceBlock), 0, st, jobs, P);
    else
      hipLaunchKernelGGL(shadow_batch_kernel<false>, dim3(gt), dim3(kTraceBlock), 0, st, jobs, P);
  }
  hipLaunchKernelGGL(resolve_batch_kernel, dim3(grid_for(total_pix)), dim3(kBlock), 0, st, jobs, nj, P, total_pix);
  return hipGetLastError();
}

namespace {
// One fiber-BSDF query per thread (rrhip_hair_bsdf).
__global__ __launch_bounds__(kBlock) void hair_bsdf_kernel(PtMaterial m, uint32_t n, const float* __restrict__ wo,
                                                          const float* __restrict__ wi, const float* __restrict__ h,
                                                          const float* __restrict__ u, float* __restrict__ f,
                                                          float* __restrict__ pdf, float* __restrict__ ws,
                                                          float* __restrict__ fs, float* __restrict__ pdfs) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const HairGeom g = hair_geom(m, v3(wo + 3 * (size_t)i), h[i]);
  V3 fv;
  float pv;
  hair_eval(m, g, v3(wi + 3 * (size_t)i), fv, pv);
  f[3 * (size_t)i] = fv.x;
  f[3 * (size_t)i + 1] = fv.y;
  f[3 * (size_t)i + 2] = fv.z;
  pdf[i] = pv;
  const float uu[4] = {u[4 * (size_t)i], u[4 * (size_t)i + 1], u[4 * (size_t)i + 2], u[4 * (size_t)i + 3]};
  V3 w, sf;
  float sp;
  const bool ok = hair_sample(m, g, uu, w, sf, sp);
  ws[3 * (size_t)i] = w.x;
  ws[3 * (size_t)i + 1] = w.y;
  ws[3 * (size_t)i + 2] = w.z;
  fs[3 * (size_t)i] = sf.x;
  fs[3 * (size_t)i + 1] = sf.y;
  fs[3 * (size_t)i + 2] = sf.z;
  pdfs[i] = ok ? sp : 0.f;
}
}  // namespace

hipError_t pt_launch_hair_bsdf(const PtMaterial& m, uint32_t n, const float* wo, const float* wi, const float* h,
                               const float* u, float* f, float* pdf, float* ws, float* fs, float* pdfs,
                               hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(hair_bsdf_kernel, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, st, m, n, wo, wi, h, u, f,
                     pdf, ws, fs, pdfs);
  return hipGetLastError();
}

hipError_t pt_launch_pcg32_draws(const uint64_t* pixel, const uint64_t* sample, uint32_t n, uint32_t count,
                                 uint32_t* out, hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(pcg32_draws_kernel, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, st, pixel, sample, n,
                     count, out);
  return hipGetLastError();
}

hipError_t pt_launch_film_image(const double* accum, const double* film, uint32_t npix, double* out, hipStream_t st) {
  hipLaunchKernelGGL(film_image_kernel, dim3((npix + kBlock - 1) / kBlock), dim3(kBlock), 0, st, accum, film, npix, out);
  return hipGetLastError();
}

hipError_t pt_launch_resolve(const PathBuffers& P, const PtParams& prm, double* accum, double* film,
                             hipStream_t st) {
  hipLaunchKernelGGL(resolve_kernel, dim3(grid_for(prm.npix)), dim3(kBlock), 0, st, P, prm, accum);
  if (film) hipLaunchKernelGGL(resolve_film_kernel, dim3(grid_for(prm.npix)), dim3(kBlock), 0, st, P, prm, film);
  return hipGetLastError();
}

}  // namespace rrhip

namespace rrhip {
namespace {

// relMSE partial sums (f64): per pixel and channel (x - r)^2 / (r^2 + eps)
// with x, r the per-pixel means of two accumulators.
__global__ __launch_bounds__(256) void relmse_kernel(const double* __restrict__ a, const double* __restrict__ r,
                                                    uint32_t npix, double eps, double* __restrict__ partial) {
  __shared__ double red[256];
  double acc = 0.0;
  const uint32_t stride = gridDim.x * blockDim.x;
  for (uint32_t p = blockIdx.x * blockDim.x + threadIdx.x; p < npix; p += stride) {
    const double* pa = a + 8 * (size_t)p;
    const double* pr = r + 8 * (size_t)p;
    const double na = pa[6] > 0.0 ? pa[6] : 1.0, nr = pr[6] > 0.0 ? pr[6] : 1.0;
    for (int c = 0; c < 3; c++) {
      const double x = pa[c] / na, ref = pr[c] / nr;
      const double d = x - ref;
      acc += d * d / (ref * ref + eps);
    }
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

}  // namespace

hipError_t pt_launch_relmse(const double* accum, const double* ref_accum, uint32_t npix, double eps,
                            double* partial, uint32_t blocks, hipStream_t st) {
  hipLaunchKernelGGL(relmse_kernel, dim3(blocks), dim3(256), 0, st, accum, ref_accum, npix, eps, partial);
  return hipGetLastError();
}

namespace {

// Per-block partial sums of the accumulators' sample counts.
__global__ __launch_bounds__(256) void count_sum_kernel(const double* __restrict__ a, uint32_t npix,
                                                        double* __restrict__ partial) {
  __shared__ double red[256];
  double acc = 0.0;
  const uint32_t stride = gridDim.x * blockDim.x;
  for (uint32_t p = blockIdx.x * blockDim.x + threadIdx.x; p < npix; p += stride) acc += a[8 * (size_t)p + 6];
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

// Adaptive stopping rule of pt/mod.rs:319-325: after the 32-sample warm-up
// a pixel stops once the 95 % confidence half-width of its mean luminance,
// 1.96 sqrt(var / n) with var the unbiased sample variance, is below
// tol * max(mean, 0.05). The moments come from the accumulator's sums
// (luminance of the rgb sum, sum of squared luminance, count), evaluated
// without fused operations so that the host can repeat the decision.
__device__ bool pixel_converged(const double* a, double tol) {
#pragma clang fp contract(off)
  const double n = a[6];
  if (n < 32.0) return false;
  const double sum = 0.2126 * a[0] + 0.7152 * a[1] + 0.0722 * a[2];
  const double mean = sum / n;
  const double var = fmax((a[7] - sum * mean) / (n - 1.0), 0.0);
  return 1.96 * sqrt(var / n) < tol * fmax(mean, 0.05);
}

constexpr uint32_t kPruneBlock = 256;

// Column c of the live list `in` (null: column = pixel) keeps sampling.
__device__ __forceinline__ bool keep_column(const double* accum, const uint32_t* in, uint32_t c, double tol,
                                            uint32_t* px) {
  *px = in ? in[c] : c;
  return !pixel_converged(accum + 8 * (size_t)*px, tol);
}

__global__ __launch_bounds__(kPruneBlock) void prune_count_kernel(const double* __restrict__ accum,
                                                                 const uint32_t* __restrict__ in, uint32_t n,
                                                                 double tol, uint32_t* __restrict__ bcount) {
  const uint32_t c = blockIdx.x * kPruneBlock + threadIdx.x;
  uint32_t px = 0;
  const bool k = c < n && keep_column(accum, in, c, tol, &px);
  const int cnt = __syncthreads_count(k);
  if (threadIdx.x == 0) bcount[blockIdx.x] = (uint32_t)cnt;
}

// Exclusive prefix of the nb block counts in place; the total into *total.
__global__ __launch_bounds__(1024) void prune_scan_kernel(uint32_t* __restrict__ bcount, uint32_t nb,
                                                         uint32_t* __restrict__ total) {
  __shared__ uint32_t part[1024];
  const uint32_t per = (nb + 1023) / 1024;
  const uint32_t b0 = threadIdx.x * per, b1 = min(nb, b0 + per);
  uint32_t sum = 0;
  for (uint32_t b = b0; b < b1; b++) sum += bcount[b];
  part[threadIdx.x] = sum;
  __syncthreads();
  for (uint32_t off = 1; off < 1024; off <<= 1) {
    const uint32_t v = threadIdx.x >= off ? part[threadIdx.x - off] : 0u;
    __syncthreads();
    part[threadIdx.x] += v;
    __syncthreads();
  }
  uint32_t run = part[threadIdx.x] - sum;
  for (uint32_t b = b0; b < b1; b++) {
    const uint32_t c = bcount[b];
    bcount[b] = run;
    run += c;
  }
  if (threadIdx.x == 1023) *total = part[1023];
}

// Writes the pixels that keep sampling, in column order.
__global__ __launch_bounds__(kPruneBlock) void prune_scatter_kernel(const double* __restrict__ accum,
                                                                   const uint32_t* __restrict__ in, uint32_t n,
                                                                   double tol, const uint32_t* __restrict__ boff,
                                                                   uint32_t* __restrict__ out) {
  __shared__ uint32_t wsum[kPruneBlock / 64];
  const uint32_t c = blockIdx.x * kPruneBlock + threadIdx.x;
  uint32_t px = 0;
  const bool k = c < n && keep_column(accum, in, c, tol, &px);
  const uint64_t m = __ballot(k);
  const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) wsum[w] = (uint32_t)__popcll(m);
  __syncthreads();
  uint32_t base = boff[blockIdx.x];
  for (uint32_t i = 0; i < w; i++) base += wsum[i];
  if (k) out[base + (uint32_t)__popcll(m & ((1ull << lane) - 1ull))] = px;
}

}  // namespace

hipError_t pt_launch_count_sum(const double* accum, uint32_t npix, double* partial, uint32_t blocks,
                               hipStream_t st) {
  hipLaunchKernelGGL(count_sum_kernel, dim3(blocks), dim3(256), 0, st, accum, npix, partial);
  return hipGetLastError();
}

hipError_t pt_launch_adaptive_prune(const double* accum, const uint32_t* in, uint32_t n, double tol,
                                    uint32_t* bcount, uint32_t* out, uint32_t* nlive, hipStream_t st) {
  const uint32_t nb = (n + kPruneBlock - 1) / kPruneBlock;
  if (nb == 0) return hipErrorInvalidValue;
  hipLaunchKernelGGL(prune_count_kernel, dim3(nb), dim3(kPruneBlock), 0, st, accum, in, n, tol, bcount);
  hipLaunchKernelGGL(prune_scan_kernel, dim3(1), dim3(1024), 0, st, bcount, nb, nlive);
  hipLaunchKernelGGL(prune_scatter_kernel, dim3(nb), dim3(kPruneBlock), 0, st, accum, in, n, tol, bcount, out);
  return hipGetLastError();
}

}  // namespace rrhip

namespace rrhip {
namespace {

// Target of training record r (path radiance `lf` at the end): the
// radiance scattered at the vertex, (L_end - L_at_vertex) / throughput,
// with the pixel estimator's firefly clamp on its luminance. Records whose
// throughput has a channel below 1e-6 carry no usable target.
__device__ __forceinline__ bool nrc_target(const NrcPathBuffers& N, size_t r, float4 lf, float clamp, float t[3]) {
  const float4 b = N.tb[r], l = N.tl[r];
  const float bb[3] = {b.x, b.y, b.z}, ll[3] = {l.x, l.y, l.z}, ff[3] = {lf.x, lf.y, lf.z};
#pragma unroll
  for (int c = 0; c < 3; c++) {
    if (!(bb[c] > 1e-6f)) return false;
    t[c] = fmaxf((ff[c] - ll[c]) / bb[c], 0.f);
    if (!isfinite(t[c])) return false;
  }
  const float lm = 0.2126f * t[0] + 0.7152f * t[1] + 0.0722f * t[2];
  if (clamp > 0.f && lm > clamp) {
    const float s = clamp / lm;
    t[0] *= s;
    t[1] *= s;
    t[2] *= s;
  }
  return true;
}

__global__ __launch_bounds__(256) void nrc_count_kernel(PathBuffers P, NrcPathBuffers N, float clamp,
                                                       uint32_t* __restrict__ cnt) {
  const uint32_t tp = blockIdx.x * blockDim.x + threadIdx.x;
  if (tp >= N.ntrain) return;
  const uint32_t nv = N.tn[tp];
  const float4 lf = P.L[N.train_base + tp];
  uint32_t c = 0;
  for (uint32_t v = 0; v < nv; v++) {
    float t[3];
    c += nrc_target(N, (size_t)tp * N.max_vertices + v, lf, clamp, t) ? 1u : 0u;
  }
  cnt[tp] = c;
}

// Exclusive prefix sum of cnt[0, n) in place (one block of 1024 threads,
// each over a contiguous chunk); the clamped total into N.counts[1].
__global__ __launch_bounds__(1024) void nrc_scan_kernel(uint32_t* __restrict__ cnt, uint32_t n, uint32_t cap,
                                                       NrcPathBuffers N, unsigned long long* __restrict__ stats) {
  __shared__ uint32_t part[1024];
  const uint32_t t = threadIdx.x;
  const uint32_t chunk = (n + 1023) / 1024;
  const uint32_t b = t * chunk, e = min(n, b + chunk);
  uint32_t s = 0;
  for (uint32_t i = b; i < e; i++) s += cnt[i];
  part[t] = s;
  __syncthreads();
  for (uint32_t off = 1; off < 1024; off <<= 1) {
    const uint32_t v = t >= off ? part[t - off] : 0u;
    __syncthreads();
    part[t] += v;
    __syncthreads();
  }
  uint32_t run = part[t] - s;  // exclusive
  for (uint32_t i = b; i < e; i++) {
    const uint32_t c = cnt[i];
    cnt[i] = run;
    run += c;
  }
  if (t == 1023) {
    N.counts[1] = min(part[1023], cap);
    stats[2] += N.counts[0];           // cache queries of the pass
    stats[3] += min(part[1023], cap);  // training samples of the pass
  }
}

__global__ __launch_bounds__(256) void nrc_scatter_kernel(PathBuffers P, NrcPathBuffers N, float clamp,
                                                         const uint32_t* __restrict__ off, uint32_t cap,
                                                         NrcQuery* __restrict__ bq, float* __restrict__ bt) {
  const uint32_t tp = blockIdx.x * blockDim.x + threadIdx.x;
  if (tp >= N.ntrain) return;
  const uint32_t nv = N.tn[tp];
  const float4 lf = P.L[N.train_base + tp];
  uint32_t o = off[tp];
  for (uint32_t v = 0; v < nv && o < cap; v++) {
    const size_t r = (size_t)tp * N.max_vertices + v;
    float t[3];
    if (!nrc_target(N, r, lf, clamp, t)) continue;
    bq[o] = N.tq[r];
    bt[3 * (size_t)o + 0] = t[0];
    bt[3 * (size_t)o + 1] = t[1];
    bt[3 * (size_t)o + 2] = t[2];
    o++;
  }
}

__global__ void nrc_set_batch_kernel(const NrcPathBuffers N, uint32_t k, uint32_t batch, uint32_t* __restrict__ n_out) {
  const uint32_t total = N.counts[1];
  const uint64_t first = (uint64_t)k * batch;
  *n_out = total > first ? (uint32_t)min<uint64_t>(total - first, batch) : 0u;
}

}  // namespace

hipError_t pt_launch_nrc_samples(const PathBuffers& P, const NrcPathBuffers& N, float clamp, uint32_t* scratch,
                                 uint32_t cap, NrcQuery* bq, float* bt, hipStream_t st) {
  if (N.ntrain == 0) return hipSuccess;
  const uint32_t g = (N.ntrain + 255) / 256;
  hipLaunchKernelGGL(nrc_count_kernel, dim3(g), dim3(256), 0, st, P, N, clamp, scratch);
  hipLaunchKernelGGL(nrc_scan_kernel, dim3(1), dim3(1024), 0, st, scratch, N.ntrain, cap, N, P.stats);
  hipLaunchKernelGGL(nrc_scatter_kernel, dim3(g), dim3(256), 0, st, P, N, clamp, scratch, cap, bq, bt);
  return hipGetLastError();
}

hipError_t pt_launch_nrc_set_batch(const NrcPathBuffers& N, uint32_t k, uint32_t batch, uint32_t* n_out,
                                   hipStream_t st) {
  hipLaunchKernelGGL(nrc_set_batch_kernel, dim3(1), dim3(1), 0, st, N, k, batch, n_out);
  return hipGetLastError();
}

}  // namespace rrhip
