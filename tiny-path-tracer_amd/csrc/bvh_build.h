// Host side of the sphere walk (walk_bvh.h): a binned-SAH tree over a scene's
// spheres, with what each sphere needs to reproduce the reference's answer.
#ifndef TPT_CSRC_BVH_BUILD_H
#define TPT_CSRC_BVH_BUILD_H

#include <algorithm>
#include <cmath>
#include <cstring>
#include <functional>
#include <vector>

#include "records.h"

namespace tptd {

struct bvh_builder {
  struct item {
    float c[3], r;
    uint32_t leaf;
  };
  std::vector<item> items;
  std::vector<bvh_node> *nodes = nullptr;

  // (plain comparisons: one minss / maxss each; the coordinates are finite)
  static float lower(float a, float b) { return a < b ? a : b; }
  static float upper(float a, float b) { return a > b ? a : b; }
  struct box {
    float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    void add(const item &s) {
      for (int k = 0; k < 3; ++k) lo[k] = lower(lo[k], s.c[k] - s.r), hi[k] = upper(hi[k], s.c[k] + s.r);
    }
    void add(const box &b) {
      for (int k = 0; k < 3; ++k) lo[k] = lower(lo[k], b.lo[k]), hi[k] = upper(hi[k], b.hi[k]);
    }
    float area() const {
      const float x = hi[0] - lo[0], y = hi[1] - lo[1], z = hi[2] - lo[2];
      return x * y + y * z + z * x;
    }
  };

  static constexpr int kBins = 16;
  // Bins along one axis, then the cheapest cut: items of bins <= *at go left.
  void cut(uint32_t first, uint32_t count, int k, float lo, float scale, float *best, int *axis, int *at) {
    box b[kBins];
    uint32_t n[kBins] = {0};
    for (uint32_t i = first; i < first + count; ++i) {
      const item &s = items[i];
      const int q = bin(s.c[k], lo, scale);
      b[q].add(s);
      ++n[q];
    }
    float right[kBins];
    box acc;
    uint32_t m = 0;
    for (int q = kBins - 1; q > 0; --q) {
      acc.add(b[q]);
      m += n[q];
      right[q] = m ? acc.area() * static_cast<float>(m) : 0.0f;
    }
    acc = box();
    m = 0;
    for (int q = 0; q + 1 < kBins; ++q) {
      acc.add(b[q]);
      m += n[q];
      if (m == 0 || m == count) continue;
      const float cost = acc.area() * static_cast<float>(m) + right[q + 1];
      if (cost < *best) *best = cost, *axis = k, *at = q;
    }
  }
  // A few items: sorted along the axis, every cut tried.
  static constexpr uint32_t kFew = 8;
  uint32_t split_few(uint32_t first, uint32_t count, int k) {
    item *v = &items[first];
    for (uint32_t i = 1; i < count; ++i) {
      const item x = v[i];
      uint32_t q = i;
      for (; q > 0 && x.c[k] < v[q - 1].c[k]; --q) v[q] = v[q - 1];
      v[q] = x;
    }
    float right[kFew];
    box acc;
    for (uint32_t i = count; --i > 0;) {
      acc.add(v[i]);
      right[i] = acc.area() * static_cast<float>(count - i);
    }
    acc = box();
    float best = INFINITY;
    uint32_t mid = 0;
    for (uint32_t i = 1; i < count; ++i) {
      acc.add(v[i - 1]);
      const float cost = acc.area() * static_cast<float>(i) + right[i];
      if (cost < best) best = cost, mid = i;
    }
    return mid;
  }
  // (limited as a float: a conversion to int is only defined in its range)
  static int bin(float c, float lo, float scale) {
    return static_cast<int>(upper(lower((c - lo) * scale, kBins - 1), 0.0f));
  }

  // Builds [first, first + count) with at most `levels` levels of nodes;
  // returns its reference and box.
  uint32_t build(uint32_t first, uint32_t count, uint32_t levels, box *out) {
    if (count == 1) {
      out->add(items[first]);
      return kBvhLeaf | items[first].leaf;
    }
    uint32_t mid = count / 2;
    if (count > 2) {
      float lo[3], hi[3];  // of the centres
      for (int k = 0; k < 3; ++k) lo[k] = hi[k] = items[first].c[k];
      for (uint32_t i = first + 1; i < first + count; ++i)
        for (int k = 0; k < 3; ++k) lo[k] = lower(lo[k], items[i].c[k]), hi[k] = upper(hi[k], items[i].c[k]);
      int wide = 0;
      for (int k = 1; k < 3; ++k)
        if (hi[k] - lo[k] > hi[wide] - lo[wide]) wide = k;
      uint32_t need = 0;  // levels a balanced split takes
      while ((1u << need) < count) ++need;
      mid = 0;
      if (need < levels && count <= kFew && hi[wide] > lo[wide]) {
        mid = split_few(first, count, wide);
      } else if (need < levels && hi[wide] > lo[wide]) {
        float best = INFINITY;
        int axis = -1, at = 0;
        // large sets along their widest axis only: the other cuts matter near the leaves
        // (no bins where the centres are so close that their scale overflows)
        for (int k = 0; k < 3; ++k)
          if (k == wide || (count <= 512 && hi[k] - lo[k] > 0.25f * (hi[wide] - lo[wide]))) {
            const float scale = kBins / (hi[k] - lo[k]);
            if (std::isfinite(scale)) cut(first, count, k, lo[k], scale, &best, &axis, &at);
          }
        if (axis >= 0) {
          const float scale = kBins / (hi[axis] - lo[axis]), l = lo[axis];
          const auto it = std::partition(items.begin() + first, items.begin() + first + count,
                                         [&](const item &s) { return bin(s.c[axis], l, scale) <= at; });
          mid = static_cast<uint32_t>(it - items.begin()) - first;
        }
      }
      if (mid == 0 || mid == count) {  // no room for an uneven split, or centres (almost) equal
        mid = count / 2;
        std::nth_element(items.begin() + first, items.begin() + first + mid, items.begin() + first + count,
                         [&](const item &a, const item &b) { return a.c[wide] < b.c[wide]; });
      }
    }
    const uint32_t id = static_cast<uint32_t>(nodes->size());
    nodes->push_back(bvh_node());
    box l, r;
    const uint32_t rl = build(first, mid, levels - 1, &l), rr = build(first + mid, count - mid, levels - 1, &r);
    bvh_node &n = (*nodes)[id];
    for (int k = 0; k < 3; ++k) n.b[k][0] = l.lo[k], n.b[k][1] = l.hi[k], n.b[k][2] = r.lo[k], n.b[k][3] = r.hi[k];
    n.ref[0] = rl, n.ref[1] = rr;
    *out = l;
    out->add(r);
    return id;
  }
};

constexpr uint32_t kMostBig = 16;  // spheres outside the tree

// The tree of a sphere-only scene, appended to nodes / leaves (slots rebased
// by sb).  Its big spheres come first among the leaves and are tested by every
// ray: the slack of the walk's bounds grows with the largest radius in the tree.
// Big is a radius above kWalkBigRadius, or, in a scene of more than 16 such
// spheres, above 4 times the 17th largest (so never more than 16 of them; with the
// fixed radius alone such scenes had no tree: 500 spheres of radius 3, 400 x 401 x
// 16, 1.91 -> 1.14 ms).  Without a usable tree (a non-finite coordinate, more than
// 2^23 spheres, boxes that tree_check.h refuses) every ray takes the general walk.
inline bvh_scene build_bvh(const tpt_flat_scene &f, uint32_t sb, std::vector<bvh_node> *nodes,
                           std::vector<bvh_leaf> *leaves) {
  bvh_scene v;
  std::memset(&v, 0, sizeof(v));
  v.root = kBvhNone;
  std::vector<bvh_leaf> all;
  all.reserve(f.n_slots);
  for (uint32_t g = f.n_segments; g-- > 0;) {  // at equal t an earlier segment wins, and the later slot within one
    std::vector<uint32_t> open;
    for (uint32_t i = f.segments[2 * g]; i < f.segments[2 * g + 1]; ++i) {
      const tpt_slot &s = f.slots[i];
      while (!open.empty() && f.slots[open.back()].a <= i) open.pop_back();
      if ((s.b >> 28) == TPT_SLOT_BOX) {
        open.push_back(i);
        continue;
      }
      bvh_leaf l;
      std::memset(&l, 0, sizeof(l));
      for (int k = 0; k < 3; ++k) l.c[k] = s.f[k];
      l.r = s.f[3];
      for (int k = 0; k < 3; ++k) {
        l.lo[k] = open.empty() ? -INFINITY : f.slots[open.back()].f[k];
        l.hi[k] = open.empty() ? INFINITY : f.slots[open.back()].f[3 + k];
      }
      l.slot = i + sb;
      l.rank = static_cast<uint32_t>(all.size());
      all.push_back(l);
    }
  }
  bool ok = !all.empty();
  uint32_t n_big = 0;
  float mag = 0.0f, rmin = INFINITY, rmax = 0.0f;
  for (const bvh_leaf &l : all) {
    for (int k = 0; k < 3; ++k) ok = ok && std::fabs(l.c[k]) < 1e15f, mag = std::fmax(mag, std::fabs(l.c[k]) + std::fabs(l.r));
    ok = ok && std::fabs(l.r) < 1e15f;
    n_big += std::fabs(l.r) > kWalkBigRadius;
  }
  if (!ok || all.size() > (1u << 23)) return v;
  float big = kWalkBigRadius;
  if (n_big > kMostBig) {
    std::vector<float> r(all.size());
    for (size_t i = 0; i < all.size(); ++i) r[i] = std::fabs(all[i].r);
    std::nth_element(r.begin(), r.begin() + kMostBig, r.end(), std::greater<float>());
    big = 4.0f * r[kMostBig];
  }
  const auto first = std::stable_partition(all.begin(), all.end(), [=](const bvh_leaf &l) { return std::fabs(l.r) > big; });
  n_big = static_cast<uint32_t>(first - all.begin());
  for (auto l = first; l != all.end(); ++l) rmin = std::fmin(rmin, std::fabs(l->r)), rmax = std::fmax(rmax, std::fabs(l->r));
  const uint32_t leaf0 = static_cast<uint32_t>(leaves->size());
  v.big0 = leaf0;
  v.n_big = n_big;
  v.ready = 1;
  v.multi = f.n_segments > 1;
  v.mag = mag;
  v.radius = std::fmax(rmax, kWalkBigRadius);
  bvh_builder b;
  b.nodes = nodes;
  b.items.reserve(all.size());
  bvh_builder::box field;
  for (uint32_t i = n_big; i < all.size(); ++i) {
    b.items.push_back({{all[i].c[0], all[i].c[1], all[i].c[2]}, std::fabs(all[i].r), leaf0 + i});
    field.add(b.items.back());
  }
  for (int k = 0; k < 3; ++k) v.lo[k] = b.items.empty() ? 0.0f : field.lo[k], v.hi[k] = b.items.empty() ? 0.0f : field.hi[k];
  v.pad = rmin > 0.0f ? kBvhPad / rmin : INFINITY;
  leaves->insert(leaves->end(), all.begin(), all.end());
  if (!b.items.empty()) {
    bvh_builder::box whole;
    v.root = b.build(0, static_cast<uint32_t>(b.items.size()), kBvhDepth, &whole);
  }
  return v;
}

}  // namespace tptd

#endif  // TPT_CSRC_BVH_BUILD_H
