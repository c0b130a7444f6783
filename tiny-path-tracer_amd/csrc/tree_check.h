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
  std::vector<uint32_t> end(f.n_slots);  // of slot i's subtree
  for (uint32_t g = 0; g < f.n_segments; ++g) {
    const uint32_t a = f.segments[2 * g], b = f.segments[2 * g + 1];
    for (uint32_t i = b; i-- > a;) {
      const tpt_slot &s = f.slots[i];
      end[i] = i + 1;
      if ((s.b >> 28) != TPT_SLOT_BOX) continue;
      const uint32_t right = s.b & TPT_PAYLOAD_MASK;
      const uint32_t child[2] = {i + 1, right == TPT_NO_RIGHT ? i + 1 : right};
      for (const uint32_t c : child) {
        if (c >= b) return false;
        if ((f.slots[c].b >> 28) != TPT_SLOT_BOX) continue;
        for (int k = 0; k < 3; ++k)
          if (!(s.f[k] <= f.slots[c].f[k] && f.slots[c].f[3 + k] <= s.f[3 + k])) return false;
      }
      if (right != TPT_NO_RIGHT && end[i + 1] != right) return false;
      end[i] = end[child[1]];
      if (end[i] != s.a) return false;
    }
    if (a < b && end[a] != b) return false;
  }
  return true;
}

}  // namespace tptd

#endif  // TPT_CSRC_TREE_CHECK_H
