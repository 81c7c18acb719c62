// Device steps of the wavefront path integrator, shared by its kernels
// (trace, shade, batches): path state, the closest-hit step, the shading
// step, shadow records and their visibility, the per-pixel resolve.
#pragma once
#include <hip/hip_runtime.h>

#include "pt_device.h"
#include "pt_hair.h"
#include "pt_kernels.h"
#include "pt_pattern.h"
#include "pt_trace.h"

namespace rrhip {
namespace pt {

constexpr int kBlock = 256;
constexpr uint32_t kMaxGrid = 4096;
// Traversal kernels: 128 lanes per block, each with a 48-entry LDS stack.
constexpr int kTraceBlock = 128;
constexpr int kTraceStack = 48;

constexpr uint32_t kFlagFromCamera = 1u << 8;
constexpr uint32_t kFlagTrain = 1u << 9;   // radiance-cache training path
constexpr uint32_t kFlagSuffix = 1u << 10; // training path past its termination vertex
// Transparent scenes: medium-stack depth (bits 11-14, 0..8) and the count of
// hull crossings / cutout pass-throughs (bits 15-19, 0..16).
constexpr uint32_t kStackShift = 11, kSkipShift = 15, kStackSkipMask = 0x1FFu << 11;
constexpr uint32_t kMaxSkips = 16;  // pt/mod.rs:32 MAX_PRESENCE_SKIPS
// Film mode: the first real hit's AOVs are recorded (bit 20); the first
// continuation has been sampled (bit 21) and was specular-like (bit 22),
// pt/mod.rs:457-470, 959-961.
constexpr uint32_t kFlagAux = 1u << 20, kFlagFirstSet = 1u << 21, kFlagFirstSpec = 1u << 22;
constexpr uint32_t kFlagKeep = kFlagTrain | kFlagSuffix | kFlagAux | kFlagFirstSet | kFlagFirstSpec;

// pt/mod.rs:33-69 MediumStack: up to 8 medium indices, 8 bits each,
// innermost at depth - 1; the atmosphere is the implicit bottom.
__device__ __forceinline__ int stack_top(uint2 st, uint32_t depth, int atmosphere) {
  if (depth == 0) return atmosphere;
  const uint32_t i = depth - 1;
  return (int)(((i < 4 ? st.x : st.y) >> (8 * (i & 3))) & 0xFFu);
}

__device__ __forceinline__ void stack_push(uint2& st, uint32_t& depth, uint32_t m) {
  if (depth >= 8) return;
  const uint32_t sh = 8 * (depth & 3);
  if (depth < 4)
    st.x = (st.x & ~(0xFFu << sh)) | (m << sh);
  else
    st.y = (st.y & ~(0xFFu << sh)) | (m << sh);
  depth++;
}

__device__ __forceinline__ void stack_pop(uint32_t& depth) {
  if (depth > 0) depth--;
}

// Places of a block's appends to up to three queues: the lanes with `next`
// and `shadow` count in the low and high half of *pair, those with `query`
// in *qcount (used when QUERY). Every lane of the block calls it; a lane's
// places are valid where its flag is set.
//
// One 64-bit atomic per block (two with QUERY): every wave of a launch
// appends at the same addresses, where an update takes about 10 ns, so one
// atomic per wave and queue bounded the shade pass: a 256 x 256 room at 16
// samples (up to 16,384 waves a pass, 7 % of the vector issue slots used)
// took 211 us a bounce, with this 67 us; device time of the frame 2.37 ->
// 1.19 ms.
template <bool QUERY>
__device__ __forceinline__ void block_append(unsigned long long* pair, uint32_t* qcount, bool next, bool shadow,
                                             bool query, uint32_t& inext, uint32_t& ishadow, uint32_t& iquery) {
  constexpr int W = kBlock / 64;
  __shared__ uint32_t s_count[W][3], s_base[W][3];
  const uint32_t w = threadIdx.x >> 6;
  const auto rank = [](uint64_t m) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
  };
  const uint64_t mn = __ballot(next), ms = __ballot(shadow), mq = QUERY ? __ballot(query) : 0;
  if ((threadIdx.x & 63u) == 0) {
    s_count[w][0] = (uint32_t)__popcll(mn);
    s_count[w][1] = (uint32_t)__popcll(ms);
    if (QUERY) s_count[w][2] = (uint32_t)__popcll(mq);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t n[3] = {0, 0, 0};
#pragma unroll
    for (int k = 0; k < W; k++)
#pragma unroll
      for (int c = 0; c < (QUERY ? 3 : 2); c++) {
        s_base[k][c] = n[c];
        n[c] += s_count[k][c];
      }
    const unsigned long long b =
        n[0] | n[1] ? atomicAdd(pair, (unsigned long long)n[0] | ((unsigned long long)n[1] << 32)) : 0;
    const uint32_t bq = QUERY && n[2] ? atomicAdd(qcount, n[2]) : 0;
#pragma unroll
    for (int k = 0; k < W; k++) {
      s_base[k][0] += (uint32_t)b;
      s_base[k][1] += (uint32_t)(b >> 32);
      if (QUERY) s_base[k][2] += bq;
    }
  }
  __syncthreads();
  inext = s_base[w][0] + rank(mn);
  ishadow = s_base[w][1] + rank(ms);
  if (QUERY) iquery = s_base[w][2] + rank(mq);
}

__device__ __forceinline__ Pcg32 load_rng(const uint4& u) {
  Pcg32 r;
  r.state = (uint64_t)u.x | ((uint64_t)u.y << 32);
  r.inc = (uint64_t)u.z | ((uint64_t)u.w << 32);
  return r;
}
__device__ __forceinline__ uint4 store_rng(const Pcg32& r) {
  return make_uint4((uint32_t)r.state, (uint32_t)(r.state >> 32), (uint32_t)r.inc, (uint32_t)(r.inc >> 32));
}

// Camera ray of (pixel, sample) into path slot `slot`.
__device__ __forceinline__ void init_path(const PtSceneView& S, const PathBuffers& P, uint32_t slot, uint32_t pixel,
                                          uint64_t sample, uint32_t flags) {
  const uint32_t x = pixel % S.cam.width, y = pixel / S.cam.width;
  // sampler.rs:24-32 per-(pixel, sample) stream; pt/mod.rs:340-356
  Pcg32 rng = Pcg32::for_pixel_sample(pixel, sample);
  V3 o, d;
  camera_ray(S.cam, x, y, rng, o, d);
  // shutter time (after the filter and lens draws) and camera motion,
  // pt/mod.rs:351-355, camera.rs:134-146
  float time = 0.f;
  if (S.motion) {
    time = rnd(rng);
    if (S.cam.has_motion_inv && time > 0.f) {
      const float* M = S.cam.motion_inv;
      float m[12];
#pragma unroll
      for (int k = 0; k < 12; k++) m[k] = ((k % 5 == 0) ? 1.f : 0.f) + (M[k] - ((k % 5 == 0) ? 1.f : 0.f)) * time;
      o = xform_point(m, o);
      d = normalize(xform_vec(m, d));
    }
  }
  P.o[slot] = make_float4(o.x, o.y, o.z, 0.f);
  P.d[slot] = make_float4(d.x, d.y, d.z, 0.f);
  P.beta[slot] = make_float4(1.f, 1.f, 1.f, time);
  P.L[slot] = make_float4(0.f, 0.f, 0.f, 0.f);
  P.prev[slot] = make_float4(o.x, o.y, o.z, 0.f);
  P.rng[slot] = store_rng(rng);
  P.flags[slot] = flags;
  P.q0[slot] = slot;
  if (P.mstk) P.mstk[slot] = make_uint2(0u, 0u);
  if (P.ld) {
    P.ld[slot] = make_float4(0.f, 0.f, 0.f, 0.f);
    P.aux0[slot] = make_float4(0.f, 0.f, 0.f, 0.f);
    P.aux1[slot] = make_float4(0.f, 0.f, 0.f, 0.f);
    P.aux_id[slot] = 0u;
  }
}

// Closest hit of the path in `slot` into hit_n / hit_m (MOTION: at the
// path's shutter time; GEO: the geometry classes the scene holds).
template <bool MOTION, int GEO, bool COUNT = false>
__device__ __forceinline__ void extend_one(const PtSceneView& S, const PathBuffers& P, uint32_t slot, uint32_t* stk,
                                           TraceCount* tc = nullptr) {
  const float4 o4 = P.o[slot], d4 = P.d[slot];
  const float time = MOTION ? P.beta[slot].w : 0.f;
  Hit h;
  if (scene_closest<kTraceBlock, MOTION, GEO, true, COUNT>(S, v3(o4.x, o4.y, o4.z), v3(d4.x, d4.y, d4.z), time,
                                                             stk, h, tc)) {
    P.hit_n[slot] = make_float4(h.n.x, h.n.y, h.n.z, h.t);
    P.hit_m[slot] = h.material | (h.front ? 0x80000000u : 0u);
    const V3 front = offset_origin(h.p, h.e), back = offset_origin(h.p, -h.e);
    float2 tw = make_float2(kNoTangent, kNoTangent);
    if ((GEO & kGeoCurves) && dot(h.tan, h.tan) > 0.5f) tw = oct_encode(h.tan);
    P.hit_front[slot] = make_float4(front.x, front.y, front.z, tw.x);
    P.hit_back[slot] = make_float4(back.x, back.y, back.z, tw.y);
    if constexpr ((GEO & kGeoSt) != 0) {  // pattern scenes: texture coordinates of the hit
      const HitSt hs = hit_st<MOTION>(S, h, time);
      P.hit_st[slot] = make_float4(hs.s, hs.t, hs.density, 0.f);
      P.hit_gs[slot] = make_float4(hs.gs.x, hs.gs.y, hs.gs.z, 0.f);
      P.hit_gt[slot] = make_float4(hs.gt.x, hs.gt.y, hs.gt.z, 0.f);
    }
  } else {
    P.hit_n[slot] = make_float4(0.f, 0.f, 0.f, -1.f);
    P.hit_m[slot] = 0;
  }
}

// pt/mod.rs:1000-1023
__device__ __forceinline__ float light_pdf_solid_angle(const PtLight& L, V3 origin, V3 hitp) {
  if (L.kind == kLightRect || L.kind == kLightDisk) {
    const V3 d = hitp - origin;
    const float dist2 = dot(d, d);
    const float cos_light = fabsf(dot(normalize(d), v3(L.n)));
    if (cos_light < 1e-9f || L.area <= 0.f) return 0.f;
    return dist2 / (cos_light * L.area);
  }
  if (L.kind == kLightSphere) {
    const V3 c = v3(L.p) - origin;
    const float dist2 = dot(c, c);
    const float sin2 = fminf(L.radius * L.radius / dist2, 1.f);
    const float cos_max = sqrtf(fmaxf(1.f - sin2, 0.f));
    const float sa = 2.f * kPi * (1.f - cos_max);
    return sa < 1e-12f ? 0.f : 1.f / sa;
  }
  return 0.f;
}

struct ShadowOut {
  V3 o, d;
  float tmax;
  float time;  // the path's shutter time
  V3 c;        // contribution before visibility (f cos L weight / pdf)
  int medium;  // transparent scenes: the medium at the ray's origin (the walk applies its transmittance)
  uint2 seed;  // transparent scenes: random stream of the blocker walk
  bool diff;   // film mode: the contribution belongs to the diffuse AOV
};

// Evaluates the BSDF towards world direction wi: f * cos(wi) and the pdf
// (the `eval` closure of pt/mod.rs:838-845).
__device__ __forceinline__ void eval_world(const PtMaterial& m, const Frame& fr, V3 wo_l, float eta, V3 wi,
                                           V3& f, float& pdf) {
  const V3 wi_l = to_local(fr, wi);
  if (wi_l.z <= 0.f) {
    f = v3(0.f, 0.f, 0.f);
    pdf = 0.f;
    return;
  }
  bsdf_eval(m, wo_l, wi_l, eta, f, pdf);
  f = f * wi_l.z;
}

// sample_light + area_light_contribution (pt/mod.rs:1032-1209), without the
// visibility test, which becomes the returned shadow ray from `origin()`
// (evaluated last, to keep it out of the BSDF evaluation's registers; with
// error-bounded origins p itself already lies outside its surface's
// rounding box). `eval(wi, f, pdf)` gives f * cos (or the phase value) and
// the pdf of the BSDF (or phase) sampling strategy for MIS. render.rs stops
// shadow rays 1e-3 short of the light; with BOUNDED the segment also stops
// short by the sampled light point's own rounding bound (projected on the
// ray through the light's cosine).
template <bool BOUNDED, class Eval>
__device__ __forceinline__ bool sample_light(const PtSceneView& S, const PtLight& L, V3 p, V3 org,
                                             const Eval& eval, float pick, Pcg32& rng, ShadowOut& out) {
  V3 f;
  float bsdf_pdf;
  const V3 rad = v3(L.radiance);
  constexpr bool bounded = BOUNDED;
  switch (L.kind) {
    case kLightPoint: {
      const V3 to = v3(L.p) - p;
      const float dist2 = fmaxf(dot(to, to), 1e-12f);
      const V3 wi = normalize(to);
      eval(wi, f, bsdf_pdf);
      if (maxc(f) <= 0.f) return false;
      out.o = org;
      out.d = wi;
      out.tmax = len(to) - 1e-3f;
      out.c = f * rad / (dist2 * pick);
      return true;
    }
    case kLightDistant: {
      const V3 base = -v3(L.p);
      V3 wi = base;
      if (L.radius > 1e-5f) {
        const float u = rnd(rng), v = rnd(rng);
        const float cos_t = 1.f - u * (1.f - L.cos_max);
        const float sin_t = sqrtf(fmaxf(1.f - cos_t * cos_t, 0.f));
        float sp, cp;
        sincosf(2.f * kPi * v, &sp, &cp);
        wi = to_world(make_frame(base), v3(sin_t * cp, sin_t * sp, cos_t));
      }
      eval(wi, f, bsdf_pdf);
      if (maxc(f) <= 0.f) return false;
      out.o = org;
      out.d = wi;
      out.tmax = 1e8f;
      out.c = f * rad / pick;
      return true;
    }
    case kLightRect:
    case kLightDisk: {
      const float u = rnd(rng), v = rnd(rng);
      V3 a, b;
      if (L.kind == kLightRect) {
        a = v3(L.e1) * u;
        b = v3(L.e2) * v;
      } else {
        const float r = sqrtf(u);
        float sn, cs;
        sincosf(2.f * kPi * v, &sn, &cs);
        a = v3(L.e1) * (r * cs);
        b = v3(L.e2) * (r * sn);
      }
      const V3 sp = v3(L.p) + a + b;
      const V3 to = sp - p;
      const float dist2 = fmaxf(dot(to, to), 1e-12f);
      const V3 wi = normalize(to);
      const float cos_light = fabsf(dot(wi, v3(L.n)));  // double-sided emitter
      if (cos_light < 1e-9f || L.area <= 0.f) return false;
      eval(wi, f, bsdf_pdf);
      if (maxc(f) <= 0.f) return false;
      const float pdf_sa = pick * dist2 / (cos_light * L.area);
      const float w = power_heuristic(pdf_sa, bsdf_pdf);
      out.o = org;
      out.d = wi;
      out.tmax = len(to) - 1e-3f;
      if (bounded) out.tmax -= L.err / fmaxf(cos_light, 1e-2f);
      out.c = f * rad * (w / pdf_sa);
      return true;
    }
    case kLightSphere: {
      const V3 tc = v3(L.p) - p;
      const float dist2 = dot(tc, tc);
      const float r = L.radius;
      if (dist2 <= r * r * 1.0001f) return false;
      const float sin2 = fminf(r * r / dist2, 1.f);
      const float cos_max = sqrtf(fmaxf(1.f - sin2, 0.f));
      const float u = rnd(rng), v = rnd(rng);
      const float cos_t = 1.f - u * (1.f - cos_max);
      const float sin_t = sqrtf(fmaxf(1.f - cos_t * cos_t, 0.f));
      float sn, cs;
      sincosf(2.f * kPi * v, &sn, &cs);
      const V3 wi = to_world(make_frame(normalize(tc)), v3(sin_t * cs, sin_t * sn, cos_t));
      eval(wi, f, bsdf_pdf);
      if (maxc(f) <= 0.f) return false;
      const float dist = sqrtf(dist2) * cos_t - sqrtf(fmaxf(r * r - dist2 * sin_t * sin_t, 0.f));
      const float pdf_sa = pick / fmaxf(2.f * kPi * (1.f - cos_max), 1e-12f);
      const float w = power_heuristic(pdf_sa, bsdf_pdf);
      out.o = org;
      out.d = wi;
      out.tmax = dist - 1e-3f;
      if (bounded) out.tmax -= L.err + sqrtf(dist2) * err_gamma(8);
      out.c = f * rad * (w / pdf_sa);
      return true;
    }
    case kLightDome: {  // pt/mod.rs:1138-1172
      const float u = rnd(rng), v = rnd(rng);
      V3 wi, lrad = rad;
      float pdf_d = kInv4Pi;
      if (S.env_rgb) {  // importance-sampled map texel
        V3 texel;
        env_sample(S, u, v, wi, texel, pdf_d);
        if (!(pdf_d > 0.f)) return false;
        lrad = texel * rad;
      } else {  // constant dome: uniform sphere, matching dome_pdf
        const float z = 1.f - 2.f * u;
        const float rr = sqrtf(fmaxf(1.f - z * z, 0.f));
        float sn, cs;
        sincosf(2.f * kPi * v, &sn, &cs);
        wi = v3(rr * cs, rr * sn, z);
      }
      const float pdf_sa = pdf_d * pick;
      eval(wi, f, bsdf_pdf);
      if (maxc(f) <= 0.f) return false;
      const float w = power_heuristic(pdf_sa, bsdf_pdf);
      out.o = org;
      out.d = wi;
      out.tmax = 1e8f;
      out.c = f * lrad * (w / pdf_sa);
      return true;
    }
    default:
      return false;
  }
}

// With NRC, the area-spread heuristic of Mueller et al. 2021 ("Real-time
// neural radiance caching for path tracing", sec. 4): a(x1..xn) =
// (sum_{i=2..n} sqrt(|x_{i-1} - x_i|^2 / (p(w_i) |cos theta_i|)))^2 against
// c * a0, a0 = |x0 - x1|^2 / (4 pi |cos theta_1|).
// One path's shading step (the per-lane part of shade_kernel): sets
// cont (continue in the next queue), shadow (+ so), shadow2 (+ se, an
// equiangular connection in a medium), query (+ nq, qbeta).
// TR: the scene is transparent (medium stack, hulls, cutouts, shadow walks).
// FILM: also the diffuse split of the radiance and the first real hit's
// AOVs (pt/mod.rs:457-470, 559-573, 690-700, 959-961).
// FIXED: render.rs's fixed push of rays off surfaces (S.ray_offset > 0)
// instead of error-bounded origins.
// HAIR: the scene has hair fibers; their curve hits scatter with the fiber
// BSDF (pt/mod.rs:738-800).
// PAT: the scene has pattern-bound materials: paths carry a ray cone (its
// spread beyond one pixel in d.w, its width in prev.w, pt/mod.rs:477-480),
// and a hit on such a material shades with the fields its patterns give
// there (pt/mod.rs:685-689, 389-440).
// MEDIA: the scene has an atmosphere or interior media (caches are never
// attached to scenes with media).
template <bool NRC, bool TR, bool FILM = false, bool FIXED = false, bool HAIR = false, bool PAT = false,
          bool MEDIA = !NRC>
__device__ __forceinline__ void shade_one(const PtSceneView& S, const PathBuffers& P, const PtParams& prm,
                                          const NrcPathBuffers& N, uint32_t slot, bool& cont, bool& shadow,
                                          bool& shadow2, ShadowOut& se, bool& query, ShadowOut& so, NrcQuery& nq,
                                          V3& qbeta) {
    const float4 o4 = P.o[slot], d4 = P.d[slot], b4 = P.beta[slot], l4 = P.L[slot], pv4 = P.prev[slot];
    const float4 hn = P.hit_n[slot];
    uint32_t flags = P.flags[slot];
    Pcg32 rng = load_rng(P.rng[slot]);
    V3 beta = v3(b4.x, b4.y, b4.z), Lr = v3(l4.x, l4.y, l4.z);
    const V3 ro = v3(o4.x, o4.y, o4.z), rd = v3(d4.x, d4.y, d4.z);
    // Surface hit point. With error-bounded origins it is the hit rebuilt
    // from the surface and pushed outside its rounding box on the ray's
    // side, which is also where reflected and shadow rays start; rays that
    // cross the surface start from its twin on the far side. render.rs's
    // fixed push takes the point along the ray.
    constexpr bool bounded = !FIXED;
    const auto hit_point = [&]() {
      if (!bounded) return ro + rd * hn.w;
      const float4 p4 = P.hit_front[slot];
      return v3(p4.x, p4.y, p4.z);
    };
    const auto far_side = [&]() {
      const float4 b4 = P.hit_back[slot];
      return v3(b4.x, b4.y, b4.z);
    };
    const float prev_pdf = o4.w;
    const V3 prev_origin = v3(pv4.x, pv4.y, pv4.z);
    const bool from_camera = (flags & kFlagFromCamera) != 0;
    uint32_t depth = flags & 0xFFu;
    float a0 = d4.w, asum = pv4.w;
    // Transparent scenes: the medium stack and the skip count
    uint2 mst = make_uint2(0u, 0u);
    uint32_t sdepth = 0, skips = 0;
    if (TR) {
      mst = P.mstk[slot];
      sdepth = (flags >> kStackShift) & 0xFu;
      skips = (flags >> kSkipShift) & 0x1Fu;
    }
    const int cur = MEDIA ? stack_top(mst, sdepth, S.atmosphere) : -1;  // the segment's medium
    // Film: radiance of this path that goes to the diffuse AOV (all of it
    // until a first continuation is sampled specular-like); aux_set: the
    // first real hit is recorded; travel: distance to it so far.
    V3 Ld = v3(0.f, 0.f, 0.f);
    const bool diff = FILM && !(flags & kFlagFirstSpec);
    bool aux_set = true;
    float travel = 0.f;
    if (FILM) {
      const float4 ld4 = P.ld[slot];
      Ld = v3(ld4.x, ld4.y, ld4.z);
      aux_set = (flags & kFlagAux) != 0;
      if (!aux_set) travel = P.aux1[slot].w;
    }
    const auto emit = [&](V3 c) {
      Lr = Lr + c;
      if (FILM && diff) Ld = Ld + c;
    };
    constexpr bool walk = TR;  // shadow rays pick up media transmittance on their walk
    bool passed = false;                   // hull crossing or cutout pass-through
    PtMaterial mres;                       // PAT: the hit's material with its patterns applied
    // The medium along this segment (pt/mod.rs:486-633): one light pick
    // per segment; for a point light an equiangular single-scatter
    // connection (pt/mod.rs:501-551); distance sampling, and at a real
    // collision NEE with the phase function (MIS-paired with the
    // equiangular strategy for point lights) and an HG continuation
    // instead of the surface.
    bool in_medium = false, absorbed = false;
    if (MEDIA && cur >= 0) {
      const PtMedium& md = S.media[cur];
      const float t_limit = hn.w < 0.f ? 1e8f : hn.w;
      const float t_seg = fminf(t_limit, md.max_distance);
      uint32_t seg_li = 0;
      float seg_pick = 0.f;
      bool has_pick = false;
      if (S.num_lights > 0) has_pick = ls_sample(S, ro + rd * fminf(t_seg * 0.5f, 50.f), rnd(rng), seg_li, seg_pick);
      const bool point_pick = has_pick && P.so2 && S.lights[seg_li].kind == kLightPoint;
      if (point_pick && t_seg > 1e-6f) {
        const PtLight& L = S.lights[seg_li];
        const V3 lp = v3(L.p);
        float pdf_eq;
        const float t_eq = equiangular_sample(ro, rd, t_seg, lp, rnd(rng), pdf_eq);
        if (pdf_eq > 1e-12f) {
          const V3 p = ro + rd * t_eq;
          const float rho = density_at(md, p);
          if (rho > 0.f) {
            const V3 tr = medium_transmittance(md, ro, rd, t_eq, rng);
            const V3 to_l = lp - p;
            const float dist2 = fmaxf(dot(to_l, to_l), 1e-12f);
            const V3 wi = normalize(to_l);
            const float ph = hg_phase(md.g, dot(rd, wi));  // hg_phase(g, -wo.wi), wo = -rd
            const float dist = sqrtf(dist2) - 1e-3f;
            const V3 vis = walk ? v3(1.f, 1.f, 1.f) : medium_transmittance(md, p, wi, dist, rng);
            if (maxc(vis) > 0.f) {
              se.medium = cur;
              const float pdf_d = distance_pdf_approx(md, t_eq, t_seg);
              const float w_eq = pdf_eq / (pdf_eq + pdf_d);
              se.o = p;
              se.d = wi;
              se.tmax = dist;
              se.c = beta * v3(md.sigma_s) * tr * vis * v3(L.radiance) *
                     (rho * ph * w_eq / (dist2 * pdf_eq * seg_pick));
              shadow2 = maxc(se.c) > 0.f;
            }
          }
        }
      }
      const MediumEvent ev = sample_distance(md, ro, rd, t_limit, beta, rng);
      beta = beta * ev.weight;
      if (ev.scatter) {
        in_medium = true;
        const V3 p = ro + rd * ev.t;
        if (FILM && !aux_set) {  // pt/mod.rs:559-570
          aux_set = true;
          flags |= kFlagAux;
          const float st[3] = {md.sigma_t[0], md.sigma_t[1], md.sigma_t[2]};
          P.aux0[slot] = make_float4(md.sigma_s[0] / fmaxf(st[0], 1e-9f), md.sigma_s[1] / fmaxf(st[1], 1e-9f),
                                     md.sigma_s[2] / fmaxf(st[2], 1e-9f), travel + ev.t);
          P.aux1[slot] = make_float4(-rd.x, -rd.y, -rd.z, 0.f);
          P.aux_id[slot] = 0u;
        }
        if (FILM) flags |= kFlagFirstSet;  // a medium scatter is a diffuse-like first continuation
        if (maxc(v3(md.emission)) > 0.f) emit(beta * v3(md.emission));
        const V3 wo = -rd;
        if (has_pick) {
          const auto eval = [&](V3 wi, V3& f, float& pdf) {
            const float ph = hg_phase(md.g, -dot(wo, wi));
            f = v3(ph, ph, ph);
            pdf = ph;
          };
          if (sample_light<bounded>(S, S.lights[seg_li], p, p, eval, seg_pick, rng, so)) {
            so.c = beta * so.c;
            so.medium = cur;
            if (!walk) so.c = so.c * medium_transmittance(md, so.o, so.d, so.tmax, rng);
            if (point_pick) {  // pt/mod.rs:583-598
              const float pdf_d = distance_pdf_approx(md, ev.t, t_seg);
              const float pdf_e = equiangular_pdf(ro, rd, t_seg, v3(S.lights[seg_li].p), ev.t);
              so.c = so.c * (pdf_d / (pdf_d + pdf_e));
            }
            shadow = maxc(so.c) > 0.f;
          }
        }
        float pdf;
        const float u1 = rnd(rng), u2 = rnd(rng);
        const V3 wi = hg_sample(md.g, wo, u1, u2, pdf);
        if (PAT) a0 += 0.4f;  // the cone widens after a scatter (pt/mod.rs:622)
        depth++;
        bool alive = true;
        if (depth >= prm.rr_start) {
          const float qq = fminf(maxc(beta), 0.95f);
          if (qq <= 0.f || rnd(rng) > qq) {
            alive = false;
          } else {
            beta = beta / qq;
          }
        }
        cont = alive && depth < prm.max_depth;
        P.o[slot] = make_float4(p.x, p.y, p.z, pdf);
        P.d[slot] = make_float4(wi.x, wi.y, wi.z, a0);
        P.prev[slot] = make_float4(p.x, p.y, p.z, asum);
        flags = depth | (flags & kFlagKeep);
      } else {
        absorbed = !(maxc(beta) > 0.f);
      }
    }
    if (in_medium || absorbed) {
      // handled above
    } else if (hn.w < 0.f) {
      // Miss: dome (with MIS) or background (pt/mod.rs:643-659).
      if (S.dome >= 0) {
        float w = 1.f;
        if (!from_camera) w = power_heuristic(prev_pdf, dome_pdf(S, rd) * ls_pmf(S, prev_origin, (uint32_t)S.dome));
        emit(beta * dome_radiance(S, S.lights[S.dome], rd) * w);
      } else {
        emit(beta * v3(S.background));
      }
    } else {
      const uint32_t hm = P.hit_m[slot];
      PtMaterial m = S.materials[hm & 0x7FFFFFFFu];
      const bool entering = (hm >> 31) != 0;
      const V3 p = hit_point();
      if constexpr (PAT) {
        // The cone grows by this segment at every surface the path does not
        // cross as a hull; bound fields follow their patterns here.
        if (!(TR && m.hull && skips < kMaxSkips)) {
          asum += hn.w * (S.pixel_spread + a0);
          if (m.bind) {
            const PatCtx pc = pat_ctx(P.hit_st[slot], P.hit_gs[slot], P.hit_gt[slot], p, v3(hn.x, hn.y, hn.z), rd,
                                      asum);
            pat_resolve_material(S, hm & 0x7FFFFFFFu, m.bind, pc, m);
          }
        }
        mres = m;
      }
      if (FILM && !aux_set) {
        if (TR && m.hull && skips < kMaxSkips) {
          travel += hn.w;  // a hull crossing is looked through (pt/mod.rs:671)
          P.aux1[slot].w = travel;
        } else {  // the first real hit, cutouts included (pt/mod.rs:688-700)
          aux_set = true;
          flags |= kFlagAux;
          const V3 ng = v3(hn.x, hn.y, hn.z);
          const V3 nf = dot(ng, rd) <= 0.f ? ng : -ng;
          P.aux0[slot] = make_float4(m.film_albedo[0], m.film_albedo[1], m.film_albedo[2], travel + hn.w);
          P.aux1[slot] = make_float4(nf.x, nf.y, nf.z, 0.f);
          P.aux_id[slot] = m.id;
        }
      }
      // Volume hull crossings toggle the medium (pt/mod.rs:662-683); a
      // cutout passes the ray with probability 1 - presence
      // (pt/mod.rs:702-710). Neither counts as a bounce.
      if (TR) {
        if (m.hull && skips < kMaxSkips) {
          passed = true;
          if (entering)
            stack_push(mst, sdepth, (uint32_t)m.interior);
          else
            stack_pop(sdepth);
        } else if (m.presence < 1.f && rnd(rng) >= m.presence && skips < kMaxSkips) {
          passed = true;
        }
        if (passed) {
          skips++;
          const V3 org = bounded ? far_side() : p + rd * S.ray_offset;
          P.o[slot] = make_float4(org.x, org.y, org.z, prev_pdf);
          if (PAT) P.prev[slot] = make_float4(pv4.x, pv4.y, pv4.z, asum);
          cont = true;
        }
      }
    }
    if (passed) {
      // the ray continues unchanged past the surface
    } else if (hn.w >= 0.f && !in_medium && !absorbed) {
      const uint32_t hm = P.hit_m[slot];
      const PtMaterial& m = PAT ? mres : S.materials[hm & 0x7FFFFFFFu];
      const bool entering = (hm >> 31) != 0;
      const V3 p = hit_point();
      const V3 ng = v3(hn.x, hn.y, hn.z);
      const V3 wo = -rd;
      const V3 nrm = dot(ng, wo) >= 0.f ? ng : -ng;
      const float eta = entering ? m.glass_ior : 1.f / m.glass_ior;
      // Emitter hit (pt/mod.rs:723-736)
      const V3 em = v3(m.emission);
      if (maxc(em) > 0.f) {
        float w = 1.f;
        if (!from_camera && m.area_light >= 0) {
          const PtLight& L = S.lights[m.area_light];
          const float pick = ls_pmf(S, prev_origin, (uint32_t)m.area_light);
          w = power_heuristic(prev_pdf, light_pdf_solid_angle(L, prev_origin, p) * pick);
        }
        emit(beta * em * w);
      }
      bool scatter = true;
      if constexpr (HAIR) {
        // A hair fiber's curve hit (the w lanes hold its tangent): NEE with
        // the fiber BSDF's value and pdf, whose shadow rays leave from the
        // viewer's side, then a sampled continuation leaving from the side
        // of the normal it points to (pt/mod.rs:738-800). The surface
        // lobes below are skipped.
        const float4 t4 = P.hit_front[slot];
        if (m.hair && t4.w < 2.f) {
          scatter = false;
          const FiberFrame ff = fiber_frame(oct_decode(t4.w, P.hit_back[slot].w), ng, wo);
          const HairGeom g = hair_geom(m, fiber_local(ff, wo), ff.h);
          if (S.num_lights > 0) {
            uint32_t li;
            float pick;
            if (ls_sample(S, p, rnd(rng), li, pick)) {
              const auto eval = [&](V3 wi, V3& f, float& pdf) { hair_eval(m, g, fiber_local(ff, wi), f, pdf); };
              if (sample_light<bounded>(S, S.lights[li], p, bounded ? p : p + ng * S.ray_offset, eval, pick, rng,
                                        so)) {
                so.c = beta * so.c;
                so.medium = cur;
                if (MEDIA && cur >= 0 && !walk)
                  so.c = so.c * medium_transmittance(S.media[cur], so.o, so.d, so.tmax, rng);
                shadow = maxc(so.c) > 0.f;
              }
            }
          }
          const float u[4] = {rnd(rng), rnd(rng), rnd(rng), rnd(rng)};
          V3 wf, fv;
          float pv;
          if (hair_sample(m, g, u, wf, fv, pv)) {
            const V3 wi = normalize(fiber_world(ff, wf));
            beta = beta * fv / pv;
            if (PAT) a0 += 0.4f;  // pt/mod.rs:780
            if (FILM && !(flags & kFlagFirstSet)) flags |= kFlagFirstSet;
            const bool out = dot(wi, ng) >= 0.f;
            const V3 org = bounded ? (out ? p : far_side()) : p + ng * (out ? S.ray_offset : -S.ray_offset);
            depth++;
            bool alive = true;
            if (depth >= prm.rr_start) {
              const float qq = fminf(maxc(beta), 0.95f);
              if (qq <= 0.f || rnd(rng) > qq) {
                alive = false;
              } else {
                beta = beta / qq;
              }
            }
            cont = alive && depth < prm.max_depth;
            P.o[slot] = make_float4(org.x, org.y, org.z, pv);
            P.d[slot] = make_float4(wi.x, wi.y, wi.z, a0);
            P.prev[slot] = make_float4(p.x, p.y, p.z, asum);
            flags = depth | (flags & kFlagKeep);
          }
        }
      }
      if constexpr (NRC) {
        const float cosv = fmaxf(fabsf(dot(ng, rd)), 1e-4f);
        const float t2 = hn.w * hn.w;
        if (from_camera) {
          a0 = t2 / (4.f * kPi * cosv);
          asum = 0.f;
        } else {
          asum += sqrtf(t2 / fmaxf(prev_pdf * cosv, 1e-30f));
        }
        const bool wide = asum * asum > N.spread * a0;
        const bool train = (flags & kFlagTrain) != 0;
        bool record = false;
        if (!train) {
          query = wide && m.has_lobes;
        } else if (!(flags & kFlagSuffix)) {
          if (wide) {
            flags |= kFlagSuffix;
            asum = 0.f;
          }
          record = m.has_lobes != 0;
        } else {
          query = wide && m.has_lobes;
          record = !query && m.has_lobes;
        }
        if (query || record) {
          nq.pos[0] = p.x;
          nq.pos[1] = p.y;
          nq.pos[2] = p.z;
          nq.roughness = m.nrc_rough;
          nq.dir[0] = wo.x;
          nq.dir[1] = wo.y;
          nq.dir[2] = wo.z;
          nq.pad0 = 0.f;
          nq.normal[0] = nrm.x;
          nq.normal[1] = nrm.y;
          nq.normal[2] = nrm.z;
          nq.pad1 = 0.f;
          nq.albedo[0] = m.nrc_albedo[0];
          nq.albedo[1] = m.nrc_albedo[1];
          nq.albedo[2] = m.nrc_albedo[2];
          nq.pad2 = 0.f;
        }
        if (record && depth < N.max_vertices) {
          const uint32_t tp = slot - N.train_base;
          const size_t r = (size_t)tp * N.max_vertices + depth;
          N.tq[r] = nq;
          N.tb[r] = make_float4(beta.x, beta.y, beta.z, 0.f);
          N.tl[r] = make_float4(Lr.x, Lr.y, Lr.z, 0.f);
          N.tn[tp] = depth + 1;
        }
        qbeta = beta;
        scatter = !query;
      }
      const Frame fr = make_frame(nrm);
      const V3 wo_l = to_local(fr, wo);
      // NEE through the light BVH (pt/mod.rs:924-956)
      if (scatter && S.num_lights > 0 && m.has_lobes) {
        uint32_t li;
        float pick;
        if (ls_sample(S, p, rnd(rng), li, pick)) {
          const auto eval = [&](V3 wi, V3& f, float& pdf) { eval_world(m, fr, wo_l, eta, wi, f, pdf); };
          if (sample_light<bounded>(S, S.lights[li], p, bounded ? p : p + nrm * S.ray_offset, eval, pick, rng, so)) {
            so.c = beta * so.c;
            so.medium = cur;
            // shadow rays through a medium carry its transmittance (or
            // pick it up on their blocker walk)
            if (MEDIA && cur >= 0 && !walk)
              so.c = so.c * medium_transmittance(S.media[cur], so.o, so.d, so.tmax, rng);
            shadow = maxc(so.c) > 0.f;
          }
        }
      }
      // BSDF continuation (pt/mod.rs:958-987)
      BsdfSample bs;
      if (scatter && bsdf_sample(m, wo_l, eta, rng, bs)) {
        const V3 wi = to_world(fr, bs.wi);
        beta = beta * bs.f * (fabsf(bs.wi.z) / bs.pdf);
        if (PAT) a0 += fminf(1.f / (1.f + bs.pdf), 0.4f);  // pt/mod.rs:967
        if (FILM && !(flags & kFlagFirstSet)) flags |= kFlagFirstSet | (bs.specular ? kFlagFirstSpec : 0u);
        const V3 org = bounded ? (bs.transmitted ? far_side() : p)
                               : p + nrm * (bs.transmitted ? -S.ray_offset : S.ray_offset);
        const V3 nd = normalize(wi);
        if (TR && bs.transmitted && m.interior >= 0) {  // pt/mod.rs:969-975
          if (entering)
            stack_push(mst, sdepth, (uint32_t)m.interior);
          else
            stack_pop(sdepth);
        }
        depth++;
        bool alive = true;
        if (depth >= prm.rr_start) {
          const float qq = fminf(maxc(beta), 0.95f);
          if (qq <= 0.f || rnd(rng) > qq) {
            alive = false;
          } else {
            beta = beta / qq;
          }
        }
        cont = alive && depth < prm.max_depth;
        P.o[slot] = make_float4(org.x, org.y, org.z, bs.pdf);
        P.d[slot] = make_float4(nd.x, nd.y, nd.z, a0);
        P.prev[slot] = make_float4(p.x, p.y, p.z, asum);
        flags = depth | (flags & kFlagKeep);  // from_camera cleared
      }
    }
    if (TR && (shadow || shadow2)) {
      so.seed = make_uint2(rng.next_u32(), rng.next_u32());
      se.seed = so.seed;
    }
    so.time = b4.w;
    se.time = b4.w;
    so.diff = diff;
    se.diff = diff;
    if (FILM) P.ld[slot] = make_float4(Ld.x, Ld.y, Ld.z, 0.f);
    if (TR) {
      P.mstk[slot] = mst;
      flags = (flags & ~kStackSkipMask) | (sdepth << kStackShift) | (skips << kSkipShift);
    }
    P.beta[slot] = make_float4(beta.x, beta.y, beta.z, b4.w);  // w: shutter time
    P.L[slot] = make_float4(Lr.x, Lr.y, Lr.z, 0.f);
    P.rng[slot] = store_rng(rng);
    P.flags[slot] = flags;
}

// Shadow record idx of path `slot`: the first ray is `a` (or `b` alone);
// with both, `b` goes to the second arrays. sc.w: bit 0 = the record has
// a second ray, bit 1 (FILM) = its contributions go to the diffuse AOV as
// well; transparent scenes: d.w holds the medium at the origin, srng the
// walk's seed.
template <bool TR, bool FILM = false>
__device__ __forceinline__ void put_shadow(const PathBuffers& P, uint32_t idx, uint32_t slot, bool s1,
                                           const ShadowOut& a, bool s2, const ShadowOut& b) {
  const ShadowOut& f = s1 ? a : b;
  const bool both = s1 && s2;
  // transparent scenes: d.w holds the medium at the origin, srng the walk's seed
  constexpr bool walk = TR;
  P.sq[idx] = slot;
  P.so[idx] = make_float4(f.o.x, f.o.y, f.o.z, f.tmax);
  P.sd[idx] = make_float4(f.d.x, f.d.y, f.d.z, walk ? (float)f.medium : 0.f);
  P.sc[idx] = make_float4(f.c.x, f.c.y, f.c.z, (both ? 1.f : 0.f) + (FILM && f.diff ? 2.f : 0.f));
  if (walk) P.srng[idx] = f.seed;
  if (P.stime) P.stime[idx] = f.time;
  if (both) {
    P.so2[idx] = make_float4(b.o.x, b.o.y, b.o.z, b.tmax);
    P.sd2[idx] = make_float4(b.d.x, b.d.y, b.d.z, walk ? (float)b.medium : 0.f);
    P.sc2[idx] = make_float4(b.c.x, b.c.y, b.c.z, 0.f);
  }
}

// The shade pass over the queue q: each path's step, then the block-wide
// append of its shadow records, continuation and cache query.
template <bool NRC, bool TR, bool MEDIA, bool FILM, bool FIXED, bool HAIR, bool PAT = false>
__device__ __forceinline__ void shade_pass(const PtSceneView& S, const PathBuffers& P, const PtParams& prm,
                                           const uint32_t* __restrict__ q, uint32_t* __restrict__ qnext,
                                           const NrcPathBuffers& N) {
  const uint32_t live = P.live(), n = live <= P.taken ? 0 : live;
  const uint32_t stride = gridDim.x * blockDim.x;
  // Block-uniform loop bound so every lane reaches the append.
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
      shade_one<NRC, TR, FILM, FIXED, HAIR, PAT, MEDIA>(S, P, prm, N, slot, cont, shadow, shadow2, se, query, so,
                                                        nq, qbeta);
    }
    uint32_t nidx, sidx, qidx;
    block_append<NRC>(P.append(), NRC ? &N.counts[0] : nullptr, cont, shadow || shadow2, query, nidx, sidx, qidx);
    if (shadow || shadow2) put_shadow<TR, FILM>(P, sidx, slot, shadow, so, shadow2, se);
    if (cont) qnext[nidx] = slot;
    if constexpr (NRC) {
      if (query) {
        N.q[qidx] = nq;
        N.q_slot[qidx] = slot;
        N.q_beta[qidx] = make_float4(qbeta.x, qbeta.y, qbeta.z, 0.f);
      }
    }
  }
}


// Fractional visibility along a shadow ray in a transparent scene
// (pt/mod.rs:1238-1306): closest hits in turn; each segment multiplies the
// transmittance of the medium on top of the stack (the origin's medium
// over the atmosphere); hulls push / pop their media, cutouts let 1 -
// presence through, anything else blocks; at most 16 blockers.
template <bool MOTION, int GEO, bool COUNT = false>
__device__ __forceinline__ V3 walk_visibility(const PtSceneView& S, V3 o, V3 d, float time, float remaining,
                                              int medium, Pcg32& rng, uint32_t* stk, TraceCount* tc = nullptr) {
  uint2 st = make_uint2(0u, 0u);
  uint32_t depth = 0;
  if (medium >= 0 && medium != S.atmosphere) stack_push(st, depth, (uint32_t)medium);
  V3 vis = v3(1.f, 1.f, 1.f);
  for (uint32_t i = 0; i < kMaxSkips; i++) {
    Hit h;
    const bool hit = scene_closest<kTraceBlock, MOTION, GEO, true, COUNT>(S, o, d, time, stk, h, tc);
    const float seg = fminf(hit ? h.t : remaining, remaining);
    const int cur = stack_top(st, depth, S.atmosphere);
    if (cur >= 0) {
      vis = vis * medium_transmittance(S.media[cur], o, d, seg, rng);
      if (maxc(vis) < 1e-4f) return v3(0.f, 0.f, 0.f);
    }
    if (!hit || h.t >= remaining) return vis;
    const PtMaterial& m = S.materials[h.material];
    if (m.hull) {
      if (h.front)
        stack_push(st, depth, (uint32_t)m.interior);
      else
        stack_pop(depth);
    } else {
      float presence = m.presence;
      if constexpr ((GEO & kGeoSt) != 0) {  // bound presence at the blocker
        if (m.bind) {
          const HitSt hs = hit_st<MOTION>(S, h, time);
          const PatCtx pc = pat_ctx(make_float4(hs.s, hs.t, hs.density, 0.f), make_float4(0.f, 0.f, 0.f, 0.f),
                                    make_float4(0.f, 0.f, 0.f, 0.f), h.p, h.n, d, 0.f);
          presence = pat_presence(S, m.bind, pc, presence);
        }
      }
      if (presence >= 1.f) return v3(0.f, 0.f, 0.f);
      vis = vis * (1.f - presence);
      if (maxc(vis) < 1e-4f) return v3(0.f, 0.f, 0.f);
    }
    if (S.ray_offset > 0.f) {
      o = o + d * (h.t + S.ray_offset);
      remaining -= h.t + S.ray_offset;
    } else {  // past the blocker: its point pushed to the far side
      const V3 on = offset_origin(h.p, -h.e);
      remaining -= dot(on - o, d);
      o = on;
    }
  }
  return vis;
}

// Shadow record i: adds each unoccluded ray's contribution to its path
// (the first ray, then the second when the record has one); with WALK the
// rays walk their blockers (transparent scenes), else one any-hit test.
template <bool WALK, bool MOTION, int GEO, bool COUNT = false>
__device__ __forceinline__ void shadow_one_t(const PtSceneView& S, const PathBuffers& P, uint32_t i, uint32_t* stk,
                                             TraceCount* tc = nullptr) {
  const float4 o = P.so[i], d = P.sd[i];
  float4 c = P.sc[i];
  const uint32_t cw = (uint32_t)c.w;  // bit 0: second ray, bit 1: diffuse AOV
  const bool two = (cw & 1u) != 0;
  const float time = MOTION ? P.stime[i] : 0.f;
  float4 c2 = make_float4(0.f, 0.f, 0.f, 0.f);
  bool v1, v2 = false;
  if constexpr (WALK) {
    const uint2 sd = P.srng[i];
    const uint64_t seed = ((uint64_t)sd.y << 32) | sd.x;
    Pcg32 r1 = Pcg32::make(seed, 1);
    const V3 t1 = walk_visibility<MOTION, GEO, COUNT>(S, v3(o.x, o.y, o.z), v3(d.x, d.y, d.z), time, o.w, (int)d.w,
                                                      r1, stk, tc);
    c = make_float4(c.x * t1.x, c.y * t1.y, c.z * t1.z, c.w);
    v1 = maxc(t1) > 0.f;
    if (two) {
      const float4 o2 = P.so2[i], d2 = P.sd2[i];
      Pcg32 r2 = Pcg32::make(seed, 2);
      const V3 t2 = walk_visibility<MOTION, GEO, COUNT>(S, v3(o2.x, o2.y, o2.z), v3(d2.x, d2.y, d2.z), time, o2.w,
                                                        (int)d2.w, r2, stk, tc);
      c2 = P.sc2[i];
      c2 = make_float4(c2.x * t2.x, c2.y * t2.y, c2.z * t2.z, 0.f);
      v2 = maxc(t2) > 0.f;
    }
  } else {
    v1 = !scene_occluded<kTraceBlock, MOTION, GEO, COUNT>(S, v3(o.x, o.y, o.z), v3(d.x, d.y, d.z), time, o.w, stk, tc);
    if (two) {
      const float4 o2 = P.so2[i], d2 = P.sd2[i];
      v2 = !scene_occluded<kTraceBlock, MOTION, GEO, COUNT>(S, v3(o2.x, o2.y, o2.z), v3(d2.x, d2.y, d2.z), time, o2.w,
                                                            stk, tc);
      c2 = P.sc2[i];
    }
  }
  if (!v1 && !v2) return;
  const uint32_t slot = P.sq[i];
  const auto add = [&](float4* buf) {
    float4 l = buf[slot];
    if (v1) {
      l.x += c.x;
      l.y += c.y;
      l.z += c.z;
    }
    if (v2) {
      l.x += c2.x;
      l.y += c2.y;
      l.z += c2.z;
    }
    buf[slot] = l;
  };
  add(P.L);
  if (P.ld && (cw & 2u)) add(P.ld);
}

template <bool QUAD>
__device__ __forceinline__ void shadow_one(const PtSceneView& S, const PathBuffers& P, uint32_t i, uint32_t* stk) {
  if (S.transparent)
    S.motion ? shadow_one_t<true, true, QUAD ? 3 : 0>(S, P, i, stk) : shadow_one_t<true, false, QUAD ? 3 : 0>(S, P, i, stk);
  else
    S.motion ? shadow_one_t<false, true, QUAD ? 3 : 0>(S, P, i, stk) : shadow_one_t<false, false, QUAD ? 3 : 0>(S, P, i, stk);
}

// Adds column col's pass samples (slots slot_base + k * npix + col) into
// its pixel's accumulator in sample order, with the firefly clamp
// (pt/mod.rs:88-95): sum of rgb, sum of rgb squared, count, and the sum of
// squared luminance that adaptive sampling reads (pt/mod.rs:314-318).
__device__ __forceinline__ void resolve_one(const PathBuffers& P, const PtParams& prm, double* accum, uint32_t col,
                                            uint32_t slot_base) {
  double s[3] = {0, 0, 0}, q[3] = {0, 0, 0}, ql = 0.0;
  for (uint32_t k = 0; k < prm.spp_pass; k++) {
    const float4 l4 = P.L[slot_base + (size_t)k * prm.npix + col];
    double l[3] = {l4.x, l4.y, l4.z};
    double lm = 0.2126 * l[0] + 0.7152 * l[1] + 0.0722 * l[2];
    if (prm.firefly_clamp > 0.f && lm > (double)prm.firefly_clamp) {
      const double sc = (double)prm.firefly_clamp / lm;
      l[0] *= sc;
      l[1] *= sc;
      l[2] *= sc;
      lm = 0.2126 * l[0] + 0.7152 * l[1] + 0.0722 * l[2];
    }
    for (int c = 0; c < 3; c++) {
      s[c] += l[c];
      q[c] += l[c] * l[c];
    }
    ql += lm * lm;
  }
  const uint32_t px = prm.live ? prm.live[col] : col;
  double* a = accum + 8 * (size_t)px;
  for (int c = 0; c < 3; c++) {
    a[c] += s[c];
    a[3 + c] += q[c];
  }
  a[6] += (double)prm.spp_pass;
  a[7] += ql;
}

// Last job whose begin (slot_begin or pix_begin) is <= x.
template <bool PIX>
__device__ __forceinline__ uint32_t find_job(const PtJob* jobs, uint32_t nj, uint32_t x) {
  uint32_t lo = 0, hi = nj;
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if ((PIX ? jobs[mid].pix_begin : jobs[mid].slot_begin) <= x)
      lo = mid;
    else
      hi = mid;
  }
  return lo;
}

inline uint32_t grid_for(uint64_t n, int block = kBlock) {
  const uint64_t b = (n + block - 1) / block;
  return (uint32_t)(b < 1 ? 1 : (b > kMaxGrid ? kMaxGrid : b));
}

}  // namespace pt
}  // namespace rrhip
