// The host build of the sphere tree (csrc/bvh_build.h) on scenes whose centres
// spread by anything from nothing to 1e14, among them spreads too small for a
// finite bin scale.  Each tree is checked: every sphere below the root once, each
// box holding its subtree, no more levels than the walk's stack takes.  And the
// check of a scene's own boxes (csrc/tree_check.h): passed by every named scene,
// failed by each way of breaking a tree.
#include <cstdio>
#include <cstdlib>
#include <random>
#include <string>

#include "../../tiny-path-tracer_amd/csrc/bvh_build.h"
#include "../../tiny-path-tracer_amd/csrc/tree_check.h"

using namespace tptd;

namespace {

struct tree {
  std::vector<bvh_node> nodes;
  std::vector<bvh_leaf> leaves;
  std::vector<int> seen;
  uint32_t deepest = 0;
  bool ok = true;

  void visit(uint32_t ref, uint32_t level, const float *lo, const float *hi) {
    if (ref & kBvhLeaf) {
      const bvh_leaf &l = leaves[ref & ~kBvhLeaf];
      ++seen[ref & ~kBvhLeaf];
      for (int k = 0; k < 3; ++k) ok = ok && lo[k] <= l.c[k] - std::fabs(l.r) && l.c[k] + std::fabs(l.r) <= hi[k];
      return;
    }
    deepest = std::max(deepest, level + 1);
    const bvh_node &n = nodes[ref];
    for (int c = 0; c < 2; ++c) {
      float a[3], b[3];
      for (int k = 0; k < 3; ++k) {
        a[k] = n.b[k][2 * c], b[k] = n.b[k][2 * c + 1];
        ok = ok && lo[k] <= a[k] && b[k] <= hi[k];
      }
      visit(n.ref[c], level + 1, a, b);
    }
  }
};

bool check(const char *name, const std::vector<tpt_slot> &slots, bool ready = true) {
  const uint32_t seg[2] = {0, static_cast<uint32_t>(slots.size())};
  tpt_flat_scene f;
  std::memset(&f, 0, sizeof(f));
  f.slots = slots.data(), f.n_slots = seg[1];
  f.segments = seg, f.n_segments = 1;
  tree t;
  const bvh_scene v = build_bvh(f, 0, &t.nodes, &t.leaves);
  t.seen.assign(t.leaves.size(), 0);
  const float lo[3] = {-INFINITY, -INFINITY, -INFINITY}, hi[3] = {INFINITY, INFINITY, INFINITY};
  if (v.ready && v.root != kBvhNone) t.visit(v.root, 0, lo, hi);
  uint32_t missing = 0;
  for (size_t i = 0; v.ready && i < t.seen.size(); ++i) missing += t.seen[i] != (i < v.n_big ? 0 : 1);
  const bool ok = t.ok && missing == 0 && t.deepest <= kBvhDepth && (v.ready != 0) == ready && v.n_big <= kMostBig;
  std::printf("%-28s %6zu spheres, ready %u, %2u levels: %s\n", name, slots.size(), v.ready, t.deepest, ok ? "ok" : "BAD");
  return ok;
}

std::vector<tpt_slot> spheres(uint32_t n, float spread, int axes, float r) {
  std::mt19937 rng(n + axes);
  std::uniform_real_distribution<float> u(-1.0f, 1.0f);
  std::vector<tpt_slot> s(n);
  for (uint32_t i = 0; i < n; ++i) {
    std::memset(&s[i], 0, sizeof(tpt_slot));
    for (int k = 0; k < axes; ++k) s[i].f[k] = spread * u(rng);
    s[i].f[3] = r;
    s[i].b = (TPT_SLOT_SPHERE << 28) | i;
  }
  return s;
}

bool regular() {
  bool ok = true;
  std::string names = tpt_scene_names();
  for (size_t a = 0; a < names.size();) {
    const size_t b = std::min(names.find(',', a), names.size());
    std::string name = names.substr(a, b - a);
    a = b + 1;
    if (name == "random_spheres_n<N>") name = "random_spheres_n3000";
    tpt_host_scene *hs = nullptr;
    if (tpt_host_scene_build(name.c_str(), 5489, &hs) != TPT_OK) continue;  // (no earth map here)
    tpt_flat_scene f;
    bool good = tpt_host_scene_flat(hs, &f) == TPT_OK && regular_trees(f);
    std::vector<tpt_slot> own(f.slots, f.slots + f.n_slots);
    f.slots = own.data();
    uint32_t tried = 0;
    for (uint32_t i = 0; i < f.n_slots && tried < 200; ++i) {
      const tpt_slot was = own[i];
      if ((was.b >> 28) != TPT_SLOT_BOX) continue;
      ++tried;
      const bool inner = i + 1 < f.n_slots && (own[i + 1].b >> 28) == TPT_SLOT_BOX;
      if (inner) {  // a bound that no longer reaches its child's
        own[i].f[1] = std::nextafter(own[i + 1].f[1], INFINITY);
        good = good && !regular_trees(f);
        own[i] = was;
        own[i].f[5] = NAN;
        good = good && !regular_trees(f);
        own[i] = was;
      }
      own[i].a = was.a - 1;
      good = good && !regular_trees(f);
      own[i] = was;
      if ((was.b & TPT_PAYLOAD_MASK) != TPT_NO_RIGHT) {
        own[i].b = was.b + 1;
        good = good && !regular_trees(f);
        own[i].b = TPT_NO_RIGHT;
        good = good && !regular_trees(f);
        own[i] = was;
      }
    }
    std::printf("%-28s %6u slots, %u boxes broken: %s\n", name.c_str(), f.n_slots, tried, good ? "ok" : "BAD");
    tpt_host_scene_destroy(hs);
    ok = ok && good;
  }
  return ok;
}

}  // namespace

int main() {
  bool ok = regular();
  char name[64];
  for (uint32_t n : {1u, 2u, 3u, 8u, 9u, 12u, 20u, 513u, 4000u})
    for (float spread : {0.0f, 1e-45f, 1e-39f, 2e-38f, 4.7e-38f, 1e-37f, 1e-20f, 1.0f, 1e14f})
      for (int axes = 1; axes <= 3; axes += 2) {
        std::snprintf(name, sizeof(name), "spread %g, %d axes", spread, axes);
        ok = check(name, spheres(n, spread, axes, 0.5f)) && ok;
      }
  std::vector<tpt_slot> s = spheres(40, 5.0f, 3, 0.5f);
  for (int i = 0; i < 20; ++i) s[i].f[0] = (i & 1) ? 1e-39f : 0.0f, s[i].f[1] = s[i].f[2] = 0.0f;
  ok = check("a cluster a denormal wide", s) && ok;
  s[3].f[1] = NAN;
  ok = check("a NaN centre", s, false) && ok;
  // radii: however large, only a few much larger than the rest stay outside
  for (float r : {2.0f, 2.5f, 300.0f}) {
    std::snprintf(name, sizeof(name), "radius %g", r);
    s = spheres(500, 1000.0f, 3, r);
    ok = check(name, s) && ok;
    for (int i = 0; i < 20; ++i) s[25 * i].f[3] = r * (3.0f + i);
    ok = check(name, s) && ok;
  }
  return ok ? 0 : 1;
}
