// Closest hit of sphere-only scenes on a tree of their own.
//
// What bounded the walk: its length.  The reference's bvh_node splits by a
// random axis, tests every box the ray crosses in pre-order, and the walk that
// repeats it visits 47 (484 spheres) to 74 slots (20k) per ray, 100 to 206 for
// the longest lane of a wave, each a dependent load.  Here a binned-SAH tree
// with both children's boxes in one 64-byte node, the nearer child first and
// boxes beyond the held hit skipped, takes 10 to 16 visits (20 to 35) and one
// sphere test per ray instead of 4 to 7.
//
// Measured, old walk -> this one: 2M rays in 20k spheres 781 -> 336 us, the
// spheres' 400x400 16 spp frame 2.48 -> 1.25 ms, textured 1600x1600 12 spp 18.5
// -> 11.5 ms, 16 pooled renders of up to 8000 spheres 11.2 -> 4.5 ms.  The tree
// costs the host about 0.3 us per sphere when the scene is created.  (Wide
// nodes and near-first order on the reference's own tree did not pay: its
// boxes overlap too much.)
//
// Why the answer is the reference's, bit for bit.  bvh_node::hit tests a
// sphere exactly when its parent node's box passes the slab test (the boxes
// above are supersets, as tree_check.h makes sure, and slab arithmetic is
// monotone in the bounds), and keeps the smallest t, at equal t the last sphere
// in its order.  So the answer is the minimum over the spheres that are hit and
// whose parent box passes: any tree may find the candidates, as long as it skips
// none.  Each candidate is then tested with the reference's arithmetic, its
// parent box too, and ties go by its rank.
//
// No candidate is skipped because every box is grown by the distance at which
// float rounding can still report a hit.  With u = 2^-24 and D the distance of
// the ray's origin from the centre, the computed b^2 - 4ac is off by at most
// 60 u a D^2 (a, the dot product and c each within 3u to 4u of their terms'
// magnitude), so it is positive only if the line passes the centre within
// sqrt(r^2 + 15 u D^2) <= r + 7.5 u D^2 / r, and <= r + sqrt(15 u) D.  The ray
// takes D to the farthest corner of the spheres' bounds.  kBvhPad and
// kBvhPadD are these constants times 1.25; 8u (|o| + M) more covers the fused
// slab arithmetic.  Along the ray, a computed root lies within 8e-4 (|t| +
// r/|d|) of the padded chord; a slack of 2^-6 (|t| + R/|d|), 19 times that for
// radii up to R, the largest in the tree, is applied at both ends.  Bigger spheres
// are tested by every ray.
//
// Rays with a direction component that is 0, tiny or huge, a NaN, or bounds
// that are not numbers take the walk of traverse.h.
#ifndef TPT_CSRC_WALK_BVH_H
#define TPT_CSRC_WALK_BVH_H

#include "walk_flat.h"

#pragma clang fp contract(off)

namespace tptd {

constexpr float kBvhPadD = 1.182e-3f;  // 1.25 sqrt(15 u)

struct bvh_best {
  float t, bound;
  uint32_t slot, rank;
};

// One sphere with the reference's arithmetic.
__device__ __forceinline__ void bvh_test(const scene_view &S, const bvh_scene &V, uint32_t leaf, v3 o, v3 d, v3 inv,
                                         float tmin, float tmax, float reach, bvh_best &best, bool &slow) {
  const float4 *q = reinterpret_cast<const float4 *>(S.bvh_leaves + leaf);
  const float4 q0 = q[0];
  float t;
  if (!sphere_t(q0.x, q0.y, q0.z, q0.w, o, d, tmin, tmax, &t)) return;
  const float4 q1 = q[1], q2 = q[2];
  const uint32_t rank = __float_as_uint(q2.w);
  if (!(t < best.t || (t == best.t && rank > best.rank))) return;
  const slot_t b{{q1.x, q1.y, q1.z, q1.w, q2.x, q2.y}, 0u, 0u};
  // With several segments a box is tested against the hits of the segments
  // before it: certain only if the box is entered before t.
  if (!slab_nn(b, o, inv, tmin, V.multi ? fminf(t, tmax) : tmax)) {
    slow = slow || (V.multi && slab_nn(b, o, inv, tmin, tmax));
    return;
  }
  best.t = t;
  best.slot = __float_as_uint(q2.z);
  best.rank = rank;
  best.bound = t + (fabsf(t) + fabsf(tmin)) * 0x1p-6f + reach;
}

// stack: this thread's column of an LDS array [kBvhDepth][STRIDE].  All lanes
// of the wave call together.  *slow: the lane needs the general walk.
template <uint32_t STRIDE>
__device__ __forceinline__ bool bvh_world(const scene_view &S, const bvh_scene &V, v3 o, v3 d, float tmin, float tmax,
                                          bool live, uint32_t *stack, hit_t *out, uint32_t *nodes, bool *slow) {
  const v3 inv{recip_rn(d.x), recip_rn(d.y), recip_rn(d.z)};
  const float mo = max3f(fabsf(o.x), fabsf(o.y), fabsf(o.z));
  const float mi = max3f(fabsf(inv.x), fabsf(inv.y), fabsf(inv.z));
  const float big = max3f(max3f(fabsf(d.x), fabsf(d.y), fabsf(d.z)), mi, mo);
  // (fmaxf drops NaNs: they are looked for in the sum)
  const float sum = ((o.x + o.y) + o.z) + ((inv.x + inv.y) + inv.z);
  bool odd = !V.ready || !(big < 0x1p40f) || sum != sum || !(tmin <= tmax);
  // growth of the boxes
  const float dx = fmaxf(fabsf(o.x - V.lo[0]), fabsf(o.x - V.hi[0])), dy = fmaxf(fabsf(o.y - V.lo[1]), fabsf(o.y - V.hi[1])),
              dz = fmaxf(fabsf(o.z - V.lo[2]), fabsf(o.z - V.hi[2]));
  const float d2 = dx * dx + dy * dy + dz * dz;
  const float pad = fminf(V.pad * d2, kBvhPadD * __builtin_amdgcn_sqrtf(d2)) + (mo + V.mag) * 0x1p-21f;
  const v3 al{(o.x + pad) * inv.x, (o.y + pad) * inv.y, (o.z + pad) * inv.z};
  const v3 ah{(o.x - pad) * inv.x, (o.y - pad) * inv.y, (o.z - pad) * inv.z};
  const float reach = 0x1p-6f * V.radius * __builtin_amdgcn_rsqf(d.x * d.x + d.y * d.y + d.z * d.z) +
                      S.walk_ulp * mi;
  const float t0 = tmin - fabsf(tmin) * 0x1p-6f - reach;
  bvh_best best{INFINITY, tmax + fabsf(tmax) * 0x1p-6f + reach, kNone, 0u};
  uint32_t visits = 0;
  const bool mine = live && !odd;
  if (mine)
    for (uint32_t k = 0; k < V.n_big; ++k) bvh_test(S, V, V.big0 + k, o, d, inv, tmin, tmax, reach, best, odd);
  uint32_t cur = mine ? V.root : kBvhNone, held = kBvhNone, sp = 0;
  auto pop = [&]() -> uint32_t { return sp ? stack[--sp * STRIDE] : kBvhNone; };
  for (;;) {
    // Inner nodes, until no lane has one to do: a lane that meets a leaf holds
    // it and goes on; a second one makes it wait.
    while (__ballot(static_cast<int32_t>(cur) >= 0) != 0ull) {
      if (static_cast<int32_t>(cur) >= 0) {
        const float4 *q = reinterpret_cast<const float4 *>(S.bvh_nodes + cur);
        const float4 x = q[0], y = q[1], z = q[2], r = q[3];
        ++visits;
        const float x0 = __builtin_fmaf(x.x, inv.x, -al.x), x1 = __builtin_fmaf(x.y, inv.x, -ah.x);
        const float y0 = __builtin_fmaf(y.x, inv.y, -al.y), y1 = __builtin_fmaf(y.y, inv.y, -ah.y);
        const float z0 = __builtin_fmaf(z.x, inv.z, -al.z), z1 = __builtin_fmaf(z.y, inv.z, -ah.z);
        const float u0 = __builtin_fmaf(x.z, inv.x, -al.x), u1 = __builtin_fmaf(x.w, inv.x, -ah.x);
        const float v0 = __builtin_fmaf(y.z, inv.y, -al.y), v1 = __builtin_fmaf(y.w, inv.y, -ah.y);
        const float w0 = __builtin_fmaf(z.z, inv.z, -al.z), w1 = __builtin_fmaf(z.w, inv.z, -ah.z);
        const float na = fmaxf(max3f(fminf(x0, x1), fminf(y0, y1), fminf(z0, z1)), t0);
        const float fa = fminf(fminf(fminf(fmaxf(x0, x1), fmaxf(y0, y1)), fmaxf(z0, z1)), best.bound);
        const float nb = fmaxf(max3f(fminf(u0, u1), fminf(v0, v1), fminf(w0, w1)), t0);
        const float fb = fminf(fminf(fminf(fmaxf(u0, u1), fmaxf(v0, v1)), fmaxf(w0, w1)), best.bound);
        const bool ha = na <= fa, hb = nb <= fb;
        const bool first = ha && (!hb || na <= nb);  // child 0 first
        const uint32_t ra = __float_as_uint(r.x), rb = __float_as_uint(r.y);
        uint32_t next = first ? ra : rb;
        if (ha && hb) stack[sp++ * STRIDE] = first ? rb : ra;
        if (!ha && !hb) next = pop();
        if (held == kBvhNone && static_cast<int32_t>(next) < 0 && next != kBvhNone) {
          held = next;
          next = pop();
        }
        cur = next;
      }
    }
    if (held != kBvhNone) {
      ++visits;
      bvh_test(S, V, held & ~kBvhLeaf, o, d, inv, tmin, tmax, reach, best, odd);
      held = kBvhNone;
    }
    if (__ballot(cur != kBvhNone) == 0ull) break;
    if (cur != kBvhNone && static_cast<int32_t>(cur) < 0) {
      held = cur;
      cur = pop();
    }
  }
  *nodes += visits;
  *slow = live && odd;
  if (mine && best.slot != kNone) {
    *out = hit_t{best.t, best.slot, kNone, S.slots[best.slot].a};
    return true;
  }
  return false;
}

// Closest hit of a sphere-only scene: the tree, then the general walk for the
// lanes that need it.  All lanes of the wave call together.  UNIFORM: every
// lane has the same scene (its tree's parameters come through scalar loads).
template <bool UNIFORM, uint32_t STRIDE>
__device__ __forceinline__ bool sphere_world(const scene_view &S, v3 o, v3 d, const ray_ctx &rc, float tmin,
                                             float tmax, bool live, uint32_t *stack, hit_t *out, uint32_t *nodes) {
  bvh_scene V;
  if (UNIFORM) {
    typedef const TPT_SCALAR bvh_scene *bvh_scene_ptr;
    bvh_scene_ptr p = (bvh_scene_ptr)(S.bvh);
    for (int k = 0; k < 3; ++k) V.lo[k] = p->lo[k], V.hi[k] = p->hi[k];
    V.pad = p->pad, V.mag = p->mag, V.radius = p->radius;
    V.root = p->root, V.big0 = p->big0, V.n_big = p->n_big, V.multi = p->multi, V.ready = p->ready;
  } else {
    V = *S.bvh;
  }
  bool slow;
  bool got = bvh_world<STRIDE>(S, V, o, d, tmin, tmax, live, stack, out, nodes, &slow);
  if (slow) got = trace_world<true>(S, o, d, rc, tmin, tmax, out, nodes);
  return got;
}

}  // namespace tptd

#endif  // TPT_CSRC_WALK_BVH_H
