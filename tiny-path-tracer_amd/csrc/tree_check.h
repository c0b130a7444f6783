// Whether a scene's slots are the trees that walk_flat.h and walk_bvh.h take
// for granted.
#ifndef TPT_CSRC_TREE_CHECK_H
#define TPT_CSRC_TREE_CHECK_H

#include <vector>

#include "../../include/tpt.h"

namespace tptd {

// True where every segment is one tree (a box's children at i + 1 and at its
// right link, its skip link at their end) and every box holds the boxes below
// it.  A primitive is then reached exactly where its innermost box is passed: the
// slab test is monotone in the bounds, so the boxes around that one pass too.
// Flattened hitables are always so; a caller's own arrays need not be, and are
// walked box by box then.
inline bool regular_trees(const tpt_flat_scene &f) {
  struct node {
    const tpt_slot *s;
    uint32_t kids;
  };
  std::vector<node> open;  // boxes around slot i
  open.reserve(64);
  for (uint32_t g = 0; g < f.n_segments; ++g) {
    const uint32_t a = f.segments[2 * g], b = f.segments[2 * g + 1];
    open.clear();
    for (uint32_t i = a; i <= b; ++i) {
      while (!open.empty() && open.back().s->a == i) {
        if (open.back().kids != ((open.back().s->b & TPT_PAYLOAD_MASK) == TPT_NO_RIGHT ? 1u : 2u)) return false;
        open.pop_back();
      }
      if (i == b) break;
      const tpt_slot &s = f.slots[i];
      const bool box = (s.b >> 28) == TPT_SLOT_BOX;
      if (!open.empty()) {
        node &p = open.back();
        if (++p.kids > 1 && (p.kids > 2 || (p.s->b & TPT_PAYLOAD_MASK) != i)) return false;
        for (int k = 0; box && k < 3; ++k)
          if (!(p.s->f[k] <= s.f[k] && s.f[3 + k] <= p.s->f[3 + k])) return false;
        if (box && s.a > p.s->a) return false;
      } else if (i != a) {
        return false;
      }
      if (box) open.push_back(node{&s, 0});
    }
    if (!open.empty()) return false;
  }
  return true;
}

}  // namespace tptd

#endif  // TPT_CSRC_TREE_CHECK_H
