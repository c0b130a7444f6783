// Closest hit of small scenes: one uniform pass over every primitive instead
// of a tree walk, with the exact reference arithmetic kept for the winner.
//
// What bounds it: VALU issue.  The sweep before it, where the wave went through
// the slots together, evaluated each slab and each rect exactly where a lane's own
// walk visits it: an IEEE division and two axis selects per rect, and a wave paid
// for the union of its lanes' visits with about a third of them idle.  Here every lane tests every
// primitive by approximations with error bounds (one reciprocal per ray and
// axis, two fused multiply-adds per rect), nothing diverges, and records come
// through the scalar cache.  Only the nearest candidate is then evaluated
// exactly (its leaf test with the reference's division, and the box of its
// parent node: an ancestor's box is a superset, as tree_check.h makes sure, whose
// slab arithmetic is monotone, so it passes when the parent's does).
//
// Measured, sweep -> this pass: Cornell 1200x1200 128 spp 41.4 -> 25.8 ms, the
// reference's box 160x120 4 spp 0.67 -> 0.31 ms, 4.2M rays with records 182 ->
// 143 us, a guided 600x600 pass 3.82 -> 3.27 ms.  A rect costs 18 instructions,
// a box of six 44.  Scenes of more than 64 slots keep their tree walks, which a
// ray leaves after a few boxes.
//
// Lanes where the approximations cannot decide take the exact walk instead
// (*slow): a candidate within its error of an edge, of t_min or t_max, or of a
// second candidate; a direction component that is 0, tiny, huge or not a
// number (the in-plane NaN rule of the reference); a winner whose exact test
// or parent box fails.  Every other primitive is then certainly missed or
// certainly farther, so the result is the reference's bit for bit.
//
// A rect whose bounds lie inside its parent box, seen through no wrapper, needs
// no box test: certain means inside by the margin, so every slab of the box is
// entered before the hit and left after it.
//
// Error bounds, u = 2^-24 and M = the scene's largest coordinate magnitude
// (local frames and wrapper offsets included): t' = fl(k - o) * (1/d) differs
// from the reference's fl(fl(k - o) / d) by at most 4u |t|; the in-plane
// coordinate fma(t', d, o) by at most 8u (|o| + M) near a bound; half-extents
// and centres add 2u M.  The margin m is 32u (1.5 |o| + M).  A box's planes are
// off by 4u |t| in time, two of them and the rounding of the coordinate by
// at most 12u (1.5 |o| + M) max|1/d|: its et.
#ifndef TPT_CSRC_WALK_FLAT_H
#define TPT_CSRC_WALK_FLAT_H

#include "traverse.h"

#pragma clang fp contract(off)

namespace tptd {

#define TPT_SCALAR __attribute__((address_space(4)))
typedef const TPT_SCALAR flat_scan *flat_scan_ptr;
typedef const TPT_SCALAR flat_group *flat_group_ptr;

// 1/d correctly rounded for 2^-100 <= |d| <= 2^100: the hardware reciprocal
// (1 ulp) and one fused Newton step (Markstein 1990; checked against the IEEE
// division for all 2^23 mantissas): 3 instructions instead of 11.  (Not a number
// where the hardware's y is infinite.)
__device__ __forceinline__ float recip_step(float d, float y) {
  return __builtin_fmaf(__builtin_fmaf(-d, y, 1.0f), y, y);
}
__device__ __forceinline__ float recip_rn(float d) { return recip_step(d, __builtin_amdgcn_rcpf(d)); }

__device__ __forceinline__ float max3f(float a, float b, float c) { return fmaxf(fmaxf(a, b), c); }

// The nearest candidates of a lane and what decides whether the nearest is certain.
struct flat_best {
  float t1, t2, t3;  // the nearest times, in order (t3: TIES only)
  float e1;          // the nearest one's excess over its bounds (certainly inside below -margin)
  uint32_t id, id2;  // records of the nearest and (TIES) the second
};

// TIES: also keeps what it takes to settle a tie of two.
template <bool TIES>
__device__ __forceinline__ void flat_offer(flat_best &b, bool pos, float t, float e, uint32_t id) {
  const float tt = pos ? t : INFINITY;
  const bool closer = tt < b.t1;
  if (TIES) {
    const uint32_t second = tt < b.t2 ? id : b.id2;
    b.id2 = closer ? b.id : second;
    b.t3 = __builtin_amdgcn_fmed3f(b.t2, b.t3, tt);
  }
  b.t2 = __builtin_amdgcn_fmed3f(b.t1, b.t2, tt);  // t1 <= t2: the median is the new second
  b.t1 = closer ? tt : b.t1;
  b.e1 = closer ? e : b.e1;
  b.id = closer ? id : b.id;
}

struct flat_rect {
  float k, c0, c1, h0, h1;
  uint32_t win;
};
__device__ __forceinline__ flat_rect flat_load(flat_scan_ptr p) {
  return flat_rect{p->k, p->c0, p->c1, p->h0, p->h1, p->win};
}

template <bool TIES, int AXIS>
__device__ __forceinline__ void flat_test(const flat_rect &p, v3 o, v3 d, v3 inv, float m, float tlo, flat_best &best) {
  const float oa = AXIS == 0 ? o.x : (AXIS == 1 ? o.y : o.z), ia = AXIS == 0 ? inv.x : (AXIS == 1 ? inv.y : inv.z);
  const float o0 = AXIS == 0 ? o.y : o.x, d0 = AXIS == 0 ? d.y : d.x;
  const float o1 = AXIS == 2 ? o.y : o.z, d1 = AXIS == 2 ? d.y : d.z;
  const float t = (p.k - oa) * ia;
  const float x = fabsf(__builtin_fmaf(t, d0, o0) - p.c0) - p.h0;
  const float y = fabsf(__builtin_fmaf(t, d1, o1) - p.c1) - p.h1;
  const float e = fmaxf(x, y);
  flat_offer<TIES>(best, (e <= m) & (t >= tlo), t, e, p.win);
}

template <bool TIES, int AXIS>
__device__ __forceinline__ flat_scan_ptr flat_rects(flat_scan_ptr p, uint32_t n, v3 o, v3 d, v3 inv, float m,
                                                    float tlo, flat_best &best) {
  // two records per wait on the scalar loads
  for (; n >= 2; n -= 2, p += 2) {
    const flat_rect a = flat_load(p), b = flat_load(p + 1);
    flat_test<TIES, AXIS>(a, o, d, inv, m, tlo, best);
    flat_test<TIES, AXIS>(b, o, d, inv, m, tlo, best);
  }
  if (n) flat_test<TIES, AXIS>(flat_load(p++), o, d, inv, m, tlo, best);
  return p;
}

// A closed box by its slabs: entered at the largest near plane n, left at the
// smallest far plane f.  A face can be hit at its plane's time only while the
// other two axes are inside, give or take their error (times et).  So the hit
// is certain when n, f and the plane next to the one that is hit are apart by
// more than et, and a miss is certain when the box is left before it is
// entered, or before t_min, by more than et or with the next plane farther
// than et.  Anything between is offered at the lowest time, which sends the
// lane to the exact walk.
template <bool TIES>
__device__ __forceinline__ void flat_box(flat_scan_ptr p, v3 o, v3 inv, float et, float tlo, flat_best &best) {
  const float x0 = (p->k - o.x) * inv.x, x1 = (p->h0 - o.x) * inv.x;
  const float y0 = (p->c0 - o.y) * inv.y, y1 = (p->h1 - o.y) * inv.y;
  const float z0 = (p->c1 - o.z) * inv.z, z1 = (p->x - o.z) * inv.z;
  const float nx = fminf(x0, x1), ny = fminf(y0, y1), nz = fminf(z0, z1);
  const float fx = fmaxf(x0, x1), fy = fmaxf(y0, y1), fz = fmaxf(z0, z1);
  const float n = max3f(nx, ny, nz), f = fminf(fminf(fx, fy), fz);
  const float n2 = __builtin_amdgcn_fmed3f(nx, ny, nz), f2 = __builtin_amdgcn_fmed3f(fx, fy, fz);
  const bool in = n >= tlo;
  const float fe = f + et;
  const bool pos = (n <= fe) & (fe >= tlo) & ((f >= tlo) | in | (f2 <= fe));
  const bool sure = (f - n > et) & ((in ? n - n2 : f2 - f) > et);
  const float t = sure ? (in ? n : f) : tlo;
  // the face: a plane of that axis, the one whose time it is
  const bool ax = t == (in ? nx : fx), ay = t == (in ? ny : fy);
  const float hi = ax ? x1 : (ay ? y1 : z1);
  const uint32_t face = (ax ? 0u : (ay ? 2u : 4u)) + (t == hi ? 1u : 0u);
  flat_offer<TIES>(best, pos, t, sure ? -INFINITY : INFINITY, p->win + face);
}

// Touches every cache line of the scene's records at once, for a kernel that
// traces one ray per thread: the loads that follow one another in the pass then
// hit the scalar cache (a 1009-ray call: 15.1 -> 9.3 us).  At most kFlatTouch
// records, half of that cache's 16 KB.
constexpr uint32_t kFlatTouch = 256;
__device__ __forceinline__ void flat_touch(const scene_view &S) {
  typedef const TPT_SCALAR uint32_t *word_ptr;
  const uint32_t ng = S.n_fgroups * (sizeof(flat_group) / 64), ns = (min(S.n_flat, kFlatTouch) * sizeof(flat_scan) + 63) / 64;
  uint32_t x = 0;
  for (uint32_t i = 0; i < ng; ++i) x |= ((word_ptr)(S.fgroups))[16 * i];
#pragma unroll 4
  for (uint32_t i = 0; i < ns; ++i) x |= ((word_ptr)(S.flat))[16 * i];
  asm volatile("" ::"s"(x));
}

// True where a lane with a zero direction component lies in the plane of a
// rect (or box face) across that axis: the reference's 0/0, accepted with t =
// NaN wherever the ray is.
__device__ __forceinline__ bool flat_in_plane(flat_scan_ptr p, uint32_t n, uint32_t n_box, v3 o, bool zx, bool zy,
                                              bool zz) {
  // (bitwise: a short circuit would branch per lane, and what is computed past
  // it would no longer count as uniform)
  bool in = false;
  const uint32_t n0 = n & 255u, n1 = (n >> 8) & 255u, n2 = (n >> 16) & 255u;
  for (uint32_t k = 0; k < n0; ++k, ++p) in |= zx & (p->k == o.x);
  for (uint32_t k = 0; k < n1; ++k, ++p) in |= zy & (p->k == o.y);
  for (uint32_t k = 0; k < n2; ++k, ++p) in |= zz & (p->k == o.z);
  p += n >> 24;
  for (uint32_t k = 0; k < n_box; ++k, ++p)
    in |= (zx & ((p->k == o.x) | (p->h0 == o.x))) | (zy & ((p->c0 == o.y) | (p->h1 == o.y))) |
          (zz & ((p->c1 == o.z) | (p->x == o.z)));
  return in;
}

// Record `id` exactly: its leaf test with the reference's arithmetic (a
// sphere's time t is exact already) and its parent's box.  sure: it is inside its
// bounds by the margin.  *order: its place in the reference's order.  False where
// the leaf is missed, or its box is not certainly passed (entered after the hit).
__device__ __forceinline__ bool flat_exact(const scene_view &S, uint32_t id, float t, v3 o, v3 d, v3 inv, float tmin,
                                           float tmax, bool lost, bool sure, hit_t *h, uint32_t *leaf,
                                           uint32_t *order, bool *rect, hit_geo *geo) {
  const float4 *q = reinterpret_cast<const float4 *>(S.fwins + id);
  const float4 q0 = q[0], q1 = q[1], q2 = q[2], q3 = q[3], q4 = q[4];
  const uint32_t word = __float_as_uint(q1.w), xf = __float_as_uint(q3.w);
  *rect = __float_as_uint(q4.x) == TPT_SLOT_RECT;
  bool got = true;
  v3 lo = o, ld = d;
  if (xf != kNone) to_local(S.xforms[xf], &lo, &ld);
  const float f[5] = {q0.x, q0.y, q0.z, q0.w, q1.x};
  if (*rect) got = rect_t(f, (word >> 28) & 3u, lo, ld, tmin, tmax, &t);
  if (geo) {
    for (int k = 0; k < 5; ++k) geo->f[k] = f[k];
    geo->kind = __float_as_uint(q4.x), geo->word = word, geo->xf = xf;
    geo->lo = lo, geo->ld = ld;
  }
  const uint32_t boxed = __float_as_uint(q3.z);
  if (boxed > (sure ? 1u : 0u) && !lost) {
    const slot_t b{{q2.x, q2.y, q2.z, q2.w, q3.x, q3.y}, 0u, 0u};
    got = got && slab_nn(b, o, inv, tmin, t + fabsf(t) * 0x1p-19f);
  }
  *h = hit_t{t, __float_as_uint(q1.y), __float_as_uint(q1.z), word};
  *leaf = __float_as_uint(q4.y);
  *order = __float_as_uint(q4.z);
  return got;
}

// A constant_medium (src/hitable.cc:98-128) bounded by a closed box.  Certain
// where the line enters the box by one face and leaves it by another, apart
// from their neighbours by more than et and from each other by more than the
// 0.0001 between the reference's two boundary queries: those then return the
// exact times of the two faces, which are computed here, and the rest of
// medium_t follows with the same arithmetic.  (With the caller's t_max in place
// of the nearest hit so far: a free path that ends beyond that hit is then
// offered beyond it.)  Undecided lanes are offered at the lowest time.  Smoke
// box 400x400 64 spp: 6.0 -> 2.1 ms against the general media walk, which
// evaluates both boundary queries rect by rect at 2 waves per SIMD.
__device__ __forceinline__ void flat_medium(const scene_view &S, flat_scan_ptr p, v3 o, v3 d, v3 wd, v3 inv,
                                            const ray_ctx &rc, float et, float tlo, float tmin, float tmax,
                                            flat_best &best) {
  const float x0 = (p->k - o.x) * inv.x, x1 = (p->h0 - o.x) * inv.x;
  const float y0 = (p->c0 - o.y) * inv.y, y1 = (p->h1 - o.y) * inv.y;
  const float z0 = (p->c1 - o.z) * inv.z, z1 = (p->x - o.z) * inv.z;
  const float nx = fminf(x0, x1), ny = fminf(y0, y1), nz = fminf(z0, z1);
  const float fx = fmaxf(x0, x1), fy = fmaxf(y0, y1), fz = fmaxf(z0, z1);
  const float n = max3f(nx, ny, nz), f = fminf(fminf(fx, fy), fz);
  const float fe = f + et;
  const bool pos = (n <= fe) & (fe >= tlo);
  if (__ballot(pos) == 0ull) return;
  const float n2 = __builtin_amdgcn_fmed3f(nx, ny, nz), f2 = __builtin_amdgcn_fmed3f(fx, fy, fz);
  const bool sure = f - n > 0.0002f + et + 0x1p-18f * (fabsf(n) + fabsf(f)) && n - n2 > et && f2 - f > et;
  float t = tlo, e = INFINITY;
  bool hit = pos;
  if (pos && sure) {
    const bool ax = n == nx, ay = n == ny, bx = f == fx, by = f == fy;
    const float k1 = ax ? (n == x0 ? p->k : p->h0) : (ay ? (n == y0 ? p->c0 : p->h1) : (n == z0 ? p->c1 : p->x));
    const float k2 = bx ? (f == x0 ? p->k : p->h0) : (by ? (f == y0 ? p->c0 : p->h1) : (f == z0 ? p->c1 : p->x));
    float t1 = (k1 - (ax ? o.x : (ay ? o.y : o.z))) / (ax ? d.x : (ay ? d.y : d.z));
    float t2 = (k2 - (bx ? o.x : (by ? o.y : o.z))) / (bx ? d.x : (by ? d.y : d.z));
    hit = false;
    // beyond t = 2048 the 0.0001 may round away: the second query then finds
    // the entry face again, and the medium is missed
    if (t1 >= static_cast<float>(static_cast<double>(t1) + 0.0001)) t2 = t1;
    if (t1 < tmin) t1 = tmin;
    if (t2 > tmax) t2 = tmax;
    if (t1 < t2) {
      const float len = sqrtf(wd.x * wd.x + wd.y * wd.y + wd.z * wd.z);
      const float inside = (t2 - t1) * len;
      typedef const TPT_SCALAR flat_win *flat_win_ptr;
      const uint4 w = medium_draws(rc, ((flat_win_ptr)(S.fwins))[p->win].leaf);
      const float hit_distance =
          static_cast<float>(static_cast<double>(-1.0f / p->density) * log(static_cast<double>(u01(w.x))));
      if (hit_distance < inside) {
        hit = true;
        t = t1 + hit_distance / len;
        e = -INFINITY;
      }
    }
  }
  flat_offer<false>(best, hit, t, e, p->win);
}

// All lanes of the wave call together.  Returns the hit of lanes that are
// live and not slow; *slow: the lane needs the exact walk.  *leaf, *geo (may be
// null): the hit's leaf id, its primitive and local ray.
//
// Zero direction components are ordinary here (lights without a sampler of
// their own send rays along x): their reciprocal is infinite as the
// reference's, a rect across that axis is at an infinite time and missed, and
// a box's slab is decided by exact comparisons, so that axis has no error.
// An origin that is NaN in every coordinate (what follows a hit at t = NaN) is
// hit by every rect at t = NaN and passes every box, whatever its direction:
// the last rect in the reference's order wins (flat_nan).
//
// MEDIA: the scene holds constant_media (all bounded by closed boxes).
//
// TIES: two rects at the same time (the bottom of a box that stands on the
// floor, seen from inside it) are both evaluated, each with its box, and the
// reference's rule applied, the smaller t, at equal t the later one.  Paths do
// not get there; for a caller's own rays it keeps such lanes off the exact walk.
template <bool TIES, bool MEDIA>
__device__ __forceinline__ bool flat_world(const scene_view &S, v3 o, v3 d, const ray_ctx &rc, float tmin, float tmax, bool live,
                                           hit_t *out, uint32_t *nodes, bool *slow, uint32_t *leaf, hit_geo *geo) {
  const bool zx = d.x == 0.0f, zy = d.y == 0.0f, zz = d.z == 0.0f;
  const v3 y{__builtin_amdgcn_rcpf(d.x), __builtin_amdgcn_rcpf(d.y), __builtin_amdgcn_rcpf(d.z)};
  const v3 inv{zx ? y.x : recip_step(d.x, y.x), zy ? y.y : recip_step(d.y, y.y), zz ? y.z : recip_step(d.z, y.z)};
  const float mo = max3f(fabsf(o.x), fabsf(o.y), fabsf(o.z));
  const float m = (1.5f * mo + S.flat_mag) * 0x1p-19f;
  // (of the hardware's reciprocals, 1 ulp off: a denormal's is infinite, and what
  // the step makes of it is no number, which a maximum would drop)
  const float my = zy ? 0.0f : fabsf(y.y);
  const float mi = max3f(zx ? 0.0f : fabsf(y.x), my, zz ? 0.0f : fabsf(y.z));
  const float big = fmaxf(max3f(fabsf(d.x), fabsf(d.y), fabsf(d.z)), fmaxf(mi, mo));
  // (fmaxf drops NaNs: they are looked for in the sum)
  const float sum = ((o.x + o.y) + o.z) + ((d.x + d.y) + d.z);
  const bool lost = o.x != o.x && o.y != o.y && o.z != o.z;
  // Every time below is finite then, so an infinite limit is as good as the
  // largest number, but for a zero direction: that one hits every rect at t = +-inf.
  const bool unlimited = !(tmax <= kFltMaxT) || !(tmin >= -kFltMaxT);
  const float t_near = fmaxf(tmin, -kFltMaxT), t_far = fminf(tmax, kFltMaxT);
  bool odd = !(big < 0x1p60f) || sum != sum || !(tmin <= tmax) || (unlimited & zx & zy & zz);
  const bool zero = live && !odd && (zx || zy || zz);
  const bool any_zero = __ballot(zero) != 0ull;
  const float tlo = t_near - fabsf(t_near) * 0x1p-19f;
  flat_best best{INFINITY, INFINITY, INFINITY, -INFINITY, kNone, kNone};
  flat_scan_ptr p = (flat_scan_ptr)(S.flat);
  flat_group_ptr groups = (flat_group_ptr)(S.fgroups);
  uint32_t visits = 0;
  for (uint32_t g = 0; g < S.n_fgroups; ++g) {
    const uint32_t n = groups[g].n, n_box = groups[g].n_box & 0xFFFFu, n_med = groups[g].n_box >> 16, nops = groups[g].nops, kinds = groups[g].kinds;
    v3 lo = o, ld = d, li = inv;
    float et = mi;
    if (nops) {
      for (uint32_t i = 0; i < nops; ++i) {
        const float p0 = groups[g].p[i][0], p1 = groups[g].p[i][1], p2 = groups[g].p[i][2];
        if (((kinds >> (2 * i)) & 3u) == TPT_XFORM_TRANSLATE) {
          lo = v3{lo.x - p0, lo.y - p1, lo.z - p2};
        } else {
          lo = v3{p1 * lo.x - p0 * lo.z, lo.y, p0 * lo.x + p1 * lo.z};
          ld = v3{p1 * ld.x - p0 * ld.z, ld.y, p0 * ld.x + p1 * ld.z};
        }
      }
      li = v3{__builtin_amdgcn_rcpf(ld.x), inv.y, __builtin_amdgcn_rcpf(ld.z)};
      et = max3f(fabsf(li.x), my, fabsf(li.z));
      odd |= !(et < 0x1p60f);
    }
    if (any_zero)  // (a zero x or z component seen through a rotation is tiny, or made the lane odd)
      odd |= flat_in_plane(p, n, n_box + n_med, lo, zero & zx & !nops, zero & zy, zero & zz & !nops);
    et *= 0.375f * m;
    p = flat_rects<TIES, 0>(p, n & 255u, lo, ld, li, m, tlo, best);
    p = flat_rects<TIES, 1>(p, (n >> 8) & 255u, lo, ld, li, m, tlo, best);
    p = flat_rects<TIES, 2>(p, (n >> 16) & 255u, lo, ld, li, m, tlo, best);
    for (uint32_t k = n >> 24; k > 0; --k, ++p) {  // spheres: exact, so certain
      float t;
      const bool h = sphere_t(p->k, p->c0, p->c1, p->h0, lo, ld, tmin, tmax, &t);
      flat_offer<TIES>(best, h, t, -INFINITY, p->win);
    }
    for (uint32_t k = n_box; k > 0; --k, ++p) flat_box<TIES>(p, lo, li, et, tlo, best);
    if (MEDIA)
      for (uint32_t k = n_med; k > 0; --k, ++p) flat_medium(S, p, lo, ld, d, li, rc, et, tlo, tmin, tmax, best);
    visits += (n & 255u) + ((n >> 8) & 255u) + ((n >> 16) & 255u) + (n >> 24) + n_box + n_med;
  }
  *nodes += live ? visits : 0u;
  // beyond t_max by more than its error: a certain miss
  bool have = best.id != kNone && !(best.t1 > t_far + fabsf(t_far) * 0x1p-19f);
  bool amb = odd;
  if (lost && tmin <= tmax) {
    best.id = S.flat_nan;
    have = best.id != kNone;
    amb = false;
  } else if (have) {
    amb = amb || best.e1 > -m || !(best.t1 > t_near + fabsf(t_near) * 0x1p-19f) ||
          !(best.t1 < t_far - fabsf(t_far) * 0x1p-19f) ||
          !((TIES ? best.t3 : best.t2) > best.t1 + fabsf(best.t1) * 0x1p-18f);
  }
  bool got = false;
  if (live && have && !amb) {
    uint32_t order, id;
    bool rect;
    got = flat_exact(S, best.id, best.t1, o, d, inv, tmin, tmax, lost, true, out, &id, &order, &rect, geo);
    if (TIES && !lost && !(best.t2 > best.t1 + fabsf(best.t1) * 0x1p-18f)) {
      hit_t h;
      uint32_t order2, id2;
      bool rect2;
      // (nothing is known of how far inside its bounds the second is; if it is missed
      // after all, the recursion decides)
      got &= flat_exact(S, best.id2, best.t2, o, d, inv, tmin, tmax, false, false, &h, &id2, &order2, &rect2, nullptr);
      got = got && rect && rect2;
      if (got && (h.t < out->t || (h.t == out->t && order2 > order))) *out = h, id = id2;
    }
    amb = !got;
    if (leaf) *leaf = id;
  }
  *slow = live && amb;
  return got;
}

// One segment (at most 64 slots) by the reference's recursion itself, the wave
// together: every slot is evaluated, last one first, so that a box finds its
// children's results (kept in scratch, at wave-uniform indexes) and combines
// them as bvh_node::hit does, `left.t < right.t ? left : right` where both hit.
// That needs no account of which boxes a lane's walk enters (a subtree under a
// missed box is dropped there), and is exact for NaN times too.  About 1400
// instructions for the Cornell box; segment_exact, a stack machine per lane,
// takes about 11000.
template <bool MEDIA>
__device__ __forceinline__ bool segment_combine(const scene_view &S, uint32_t start, uint32_t end, v3 o, v3 d, v3 inv,
                                                const ray_ctx &rc, float tmin, float tmax, hit_t *out) {
  float ts[64];
  uint32_t ids[64];  // slot - start, and the list entry + 1 from bit 8
  unsigned long long hits = 0;
  for (uint32_t i = end; i-- > start;) {
    const slot_t s = load_slot(&S.slots[i]);
    const uint32_t kind = s.b >> 28, k = i - start;
    bool have;
    float t = 0.0f;
    uint32_t id = k;
    if (kind == TPT_SLOT_BOX) {
      const uint32_t right = s.b & TPT_PAYLOAD_MASK;
      const bool two = right != TPT_NO_RIGHT;
      const uint32_t kr = two ? right - start : k + 1;
      const float tl = ts[k + 1], tr = ts[kr];
      const bool hl = (hits >> (k + 1)) & 1ull, hr = two && ((hits >> kr) & 1ull);
      const bool left = hl && (!hr || tl < tr);
      have = slab(s, o, inv, tmin, tmax) && (hl || hr);
      t = left ? tl : tr;
      id = left ? ids[k + 1] : ids[kr];
    } else {
      uint32_t entry, mat;
      have = leaf_t<false, MEDIA>(S, s, kind, o, d, rc, tmin, tmax, &t, &entry, &mat);
      if (kind == TPT_SLOT_LIST && have) id |= (entry - s.a + 1) << 8;
    }
    ts[k] = t;
    ids[k] = id;
    hits |= have ? 1ull << k : 0ull;
  }
  const bool got = hits & 1ull;
  if (got) {
    const uint32_t slot = start + (ids[0] & 255u), e = ids[0] >> 8;
    const uint32_t a = S.slots[slot].a;
    *out = hit_t{ts[0], slot, e ? a + e - 1 : kNone, e ? S.entries[a + e - 1].a : a};
  }
  return got;
}

// Closest hit of a small scene: the uniform pass, then the exact recursion for
// the lanes that need it.  All lanes of the wave call together.
template <bool TIES = false, bool MEDIA = false>
__device__ __forceinline__ bool small_world(const scene_view &S, v3 o, v3 d, const ray_ctx &rc, float tmin, float tmax,
                                            hit_t *out, uint32_t *nodes, bool live, uint32_t *leaf = nullptr,
                                            hit_geo *geo = nullptr) {
  bool slow;
  bool got = flat_world<TIES, MEDIA>(S, o, d, rc, tmin, tmax, live, out, nodes, &slow, leaf, geo);
  if (__ballot(slow) != 0ull) {
    const v3 inv{1.0f / d.x, 1.0f / d.y, 1.0f / d.z};
    hit_t best{0.0f, kNone, kNone, 0};
    float cur = tmax;
    bool any = false;
    for (uint32_t g = 0; g < S.n_segments; ++g) {
      const uint32_t start = S.segments[2 * g], end = S.segments[2 * g + 1];
      hit_t h;
      if (start < end && segment_combine<MEDIA>(S, start, end, o, d, inv, rc, tmin, cur, &h)) {
        best = h;
        cur = h.t;
        any = true;
      }
    }
    if (slow) {
      got = any;
      *out = best;
      if (leaf && any) *leaf = leaf_id(S, best);
      if (geo && any) {
        const slot_t s = load_slot(&S.slots[best.slot]);
        for (int k = 0; k < 5; ++k) geo->f[k] = s.f[k];
        geo->kind = s.b >> 28, geo->word = s.a, geo->xf = kNone;
        geo->lo = o, geo->ld = d;
        if (best.entry != kNone) {
          const tpt_entry en = S.entries[best.entry];
          for (int k = 0; k < 5; ++k) geo->f[k] = en.f[k];
          geo->kind = en.b, geo->word = en.a, geo->xf = en.xform;
          if (en.xform != kNone) to_local(S.xforms[en.xform], &geo->lo, &geo->ld);
        }
      }
    }
  }
  return got;
}

}  // namespace tptd

#endif  // TPT_CSRC_WALK_FLAT_H
