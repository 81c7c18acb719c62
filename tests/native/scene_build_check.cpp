// Looks into the host build of a path-tracing scene for
// test_scene_build.py: what the instance hierarchy holds, how deep a
// traversal's stack gets in it, and a plain restatement of the box builder.
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <random>
#include <string>
#include <vector>

#include "bvh_build.h"
#include "pt_scene.h"

using namespace rrhip;

namespace {

PtSceneHost g_scene;

struct Box {
  float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
  void grow(const Box& b) {
    for (int a = 0; a < 3; a++) {
      lo[a] = std::min(lo[a], b.lo[a]);
      hi[a] = std::max(hi[a], b.hi[a]);
    }
  }
  double area() const {
    const double x = (double)hi[0] - lo[0], y = (double)hi[1] - lo[1], z = (double)hi[2] - lo[2];
    return x < 0 || y < 0 || z < 0 ? 0.0 : 2.0 * (x * y + y * z + z * x);
  }
};

// Leaves of the binned surface-area build in order, as (first, count) runs
// of `ids`: every boundary of every axis is priced.
void split(const std::vector<Box>& pb, const BuildParams& p, uint32_t* ids, uint32_t count, uint32_t at,
           std::vector<std::pair<uint32_t, uint32_t>>& leaves) {
  if (count <= (uint32_t)p.max_leaf) {
    leaves.push_back({at, count});
    return;
  }
  const auto mid = [&](uint32_t q, int a) { return 0.5f * (pb[q].lo[a] + pb[q].hi[a]); };
  int axis = -1, bin = 0;
  double best = INFINITY;
  float lo[3], scale[3];
  const auto bin_of = [&](uint32_t q, int a) {
    return std::min(std::max((int)((mid(q, a) - lo[a]) * scale[a]), 0), p.bins - 1);
  };
  for (int a = 0; a < 3; a++) {
    float hi = -INFINITY;
    lo[a] = INFINITY;
    for (uint32_t k = 0; k < count; k++) {
      lo[a] = std::min(lo[a], mid(ids[k], a));
      hi = std::max(hi, mid(ids[k], a));
    }
    if (!(hi - lo[a] > 0.f)) continue;
    scale[a] = (float)p.bins / (hi - lo[a]);
    for (int b = 0; b < p.bins - 1; b++) {
      Box side[2];
      uint32_t n[2] = {0, 0};
      for (uint32_t k = 0; k < count; k++) {
        const int r = bin_of(ids[k], a) > b;
        side[r].grow(pb[ids[k]]);
        n[r]++;
      }
      const double cost = side[0].area() * n[0] + side[1].area() * n[1];
      if (n[0] && n[1] && cost < best) {
        best = cost;
        axis = a;
        bin = b;
      }
    }
  }
  uint32_t left = 0;
  if (axis >= 0)
    left = (uint32_t)(std::partition(ids, ids + count, [&](uint32_t q) { return bin_of(q, axis) <= bin; }) - ids);
  if (left == 0 || left == count) left = count / 2;
  split(pb, p, ids, left, at, leaves);
  split(pb, p, ids + left, count - left, at + left, leaves);
}

}  // namespace

extern "C" {

// Builds `d`; returns the number of instances, or -1.
int check_build(const rrhip_scene_desc* d) {
  std::string err;
  g_scene = PtSceneHost{};
  return build_pt_scene(*d, &g_scene, &err) ? (int)g_scene.insts.size() : -1;
}

uint32_t check_stack_need() { return g_scene.stack_need; }

// Per instance in leaf order: its leaf's box (lo, hi), its placement and
// its geometry. Returns the most instances in a leaf.
int check_leaves(float* boxes, float* fwd, uint32_t* geometry) {
  uint32_t most = 0;
  std::vector<uint32_t> todo = {0};
  while (!todo.empty()) {
    const Node2 n = g_scene.nodes[todo.back()];
    todo.pop_back();
    const float b[2][6] = {{n.c0_lox, n.c0_loy, n.c0_loz, n.c0_hix, n.c0_hiy, n.c0_hiz},
                           {n.c1_lox, n.c1_loy, n.c1_loz, n.c1_hix, n.c1_hiy, n.c1_hiz}};
    const uint32_t ref[2] = {n.ref0, n.ref1}, cnt[2] = {n.cnt0, n.cnt1};
    for (int k = 0; k < 2; k++) {
      if (cnt[k] == 0) todo.push_back(ref[k]);
      most = std::max(most, cnt[k]);
      for (uint32_t i = ref[k]; i < ref[k] + cnt[k]; i++) std::memcpy(boxes + 6 * i, b[k], sizeof(b[k]));
    }
  }
  for (size_t i = 0; i < g_scene.insts.size(); i++) {
    std::memcpy(fwd + 12 * i, &g_scene.inst_fwd[12 * i], 12 * sizeof(float));
    geometry[i] = g_scene.insts[i].mesh;
  }
  return (int)most;
}

// The most entries a lane's stack holds over `walks` traversals that hit
// every child (miss = 0) or lose each with probability `miss`, the nearer
// interior child drawn at random or, in the first two, always the same: the
// pushes and pops of the device's InstTrace.
int check_stack_use(int walks, double miss, uint64_t seed) {
  std::mt19937_64 rng(seed);
  std::uniform_real_distribution<double> u(0.0, 1.0);
  struct Entry {
    bool inst;
    uint32_t ref, cnt;
  };
  int most = 0;
  for (int w = 0; w < walks; w++) {
    std::vector<Entry> st;
    const auto push = [&](Entry e) {
      st.push_back(e);
      most = std::max(most, (int)st.size());
    };
    int base = -1;
    bool have = true;
    uint32_t node = 0;
    for (;;) {
      if (!have) {
        if (base >= 0 && (int)st.size() == base) base = -1;
        if (st.empty()) break;
        const Entry e = st.back();
        st.pop_back();
        if (e.inst) {
          if (e.cnt > 1) push({true, e.ref + 1, e.cnt - 1});
          node = g_scene.meshes[g_scene.insts[e.ref].mesh].root;
          if (node == 0xFFFFFFFFu) continue;
          base = (int)st.size();
        } else {
          node = e.ref;
        }
      }
      const Node2 n = g_scene.nodes[node];
      const bool h0 = u(rng) >= miss, h1 = u(rng) >= miss;
      if (base < 0) {
        if (h0 && n.cnt0) push({true, n.ref0, n.cnt0});
        if (h1 && n.cnt1) push({true, n.ref1, n.cnt1});
      }
      const bool in0 = h0 && !n.cnt0, in1 = h1 && !n.cnt1;
      const bool first0 = w == 0 || (w > 1 && u(rng) < 0.5);
      have = in0 || in1;
      if (in0 && in1) push({false, first0 ? n.ref1 : n.ref0, 0});
      if (have) node = in0 && (first0 || !in1) ? n.ref0 : n.ref1;
    }
  }
  return most;
}

// 1 if build_box_bvh makes the leaves of the plain restatement.
int check_box_build(const float* boxes, uint32_t n, int bins, int max_leaf) {
  BuildParams p;
  p.bins = bins;
  p.max_leaf = max_leaf;
  BuiltBvh out;
  std::vector<uint32_t> order, ids(n);
  std::string err;
  if (!build_box_bvh(boxes, n, p, &out, &order, &err)) return 0;
  std::vector<Box> pb(n);
  for (uint32_t i = 0; i < n; i++) {
    ids[i] = i;
    std::memcpy(pb[i].lo, boxes + 6 * i, sizeof(pb[i].lo));
    std::memcpy(pb[i].hi, boxes + 6 * i + 3, sizeof(pb[i].hi));
  }
  std::vector<std::pair<uint32_t, uint32_t>> want, got;
  split(pb, p, ids.data(), n, 0, want);
  for (const Node2& b : out.nodes) {
    if (b.cnt0) got.push_back({b.ref0, b.cnt0});
    if (b.cnt1) got.push_back({b.ref1, b.cnt1});
  }
  std::sort(got.begin(), got.end());
  got.erase(std::unique(got.begin(), got.end()), got.end());  // a lone leaf is both children of the root
  return order == ids && got == want;
}

}  // extern "C"
