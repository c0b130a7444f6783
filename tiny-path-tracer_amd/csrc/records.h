// Plain records that the host prepares for the uniform pass (walk_flat.h) and
// the sphere walk (walk_bvh.h); no device code, so host programs include it too.
#ifndef TPT_CSRC_RECORDS_H
#define TPT_CSRC_RECORDS_H

#include <cstdint>

#include "../../include/tpt.h"

namespace tptd {

// What the uniform pass of walk_flat.h reads of a small scene's primitives, 32
// bytes each, through scalar loads.  rect: plane k, in-plane centres c0, c1
// and half-extents h0, h1.  sphere: centre (k, c0, c1), radius h0.  box (six
// rects of one list that close a box): low corner (k, c0, c1), high corner
// (h0, h1, x).  medium (bounded by a closed box): the box and its density.  win: its record in flat_wins (a box: of its low x face, then
// high x, low y, high y, low z, high z).
struct flat_scan {
  float k, c0, c1, h0, h1, x;
  uint32_t win;
  float density;
};
// What its winner needs, 80 bytes.
struct flat_win {
  float f[5];                 // primitive parameters as in tpt_slot
  uint32_t slot, entry, mat;  // as in hit_t
  float box[6];               // the innermost box around it
  uint32_t boxed;             // 0: there is none; 1: it is passed whenever the winner is certain; 2: it is to be tested
  uint32_t xform, kind, leaf;  // wrapper chain or ~0u; TPT_SLOT_RECT, _SPHERE or _MEDIUM; leaf id
  uint32_t order, pad;         // its place in the order of segments, slots and entries
};
// Primitives seen through one wrapper chain, in this order: rects by normal
// axis (counts in bits 0-7, 8-15, 16-23 of n), spheres (24-31), boxes and
// media (low and high half of n_box);
// and the chain itself (nops 0: none), so that one load fetches all of it.
struct flat_group {
  uint32_t n, n_box, nops, kinds;
  float p[TPT_XFORM_MAX_OPS][3];
};

// The tree of a sphere-only scene (walk_bvh.h).  A node holds both children's
// boxes, b[axis] = (low, high of child 0, low, high of child 1), and their
// references: a node, or kBvhLeaf | leaf.  A leaf: the sphere, its parent box
// in the reference's tree (infinite: none), its slot, and its rank among equal t.
constexpr uint32_t kBvhLeaf = 0x80000000u, kBvhNone = 0xFFFFFFFFu;
constexpr uint32_t kBvhDepth = 24;  // most levels of nodes (2^24 spheres fit a balanced one)
constexpr float kWalkBigRadius = 2.0f;  // spheres above it are tested by every ray (but see build_bvh)
constexpr float kBvhPad = 5.6e-7f;  // 1.25 * 7.5 u
struct bvh_node {
  float b[3][4];
  uint32_t ref[2], pad[2];
};
struct bvh_leaf {
  float c[3], r, lo[3], hi[3];
  uint32_t slot, rank;
};
struct bvh_scene {
  float lo[3], hi[3];  // bounds of the spheres in the tree
  float pad, mag;      // kBvhPad over their smallest radius; the largest coordinate magnitude
  uint32_t root, big0, n_big;  // big spheres: leaves [big0, big0 + n_big)
  uint32_t multi, ready;       // more than one segment; a tree was built
  float radius;                // none in the tree has a larger one
  uint32_t unused[2];
};

}  // namespace tptd

#endif  // TPT_CSRC_RECORDS_H
