// Plain renders in one launch per pass: every lane carries one path at a time
// through all its bounces in registers, and takes the next camera ray when it
// ends.
//
// What bounded the bounce loop (k_trace + k_shade per bounce): each segment
// moved 228 B of path records through HBM, every wave waited for three
// dependent queue atomics per step, and a small frame waited for a launch pair
// per bounce.  Here a segment moves nothing and a path 12 B (its result).
// What is left is the issue of the walk and of the shading; material classes
// of one wave run one after the other, which costs less than sorting them
// through memory did.  Camera rays are generated 64 at a time by the whole
// wave into an LDS pool from which ended lanes are refilled: ray generation
// (two Philox blocks and three double divisions) never runs for a few lanes.
// Measured, bounce loop -> this kernel: Cornell 1200x1200 128 spp 48.8 -> 41.4
// ms, random spheres 400x400 16 spp 3.39 -> 2.51 ms, 16 pooled renders of up
// to 8000 spheres 14.3 -> 11.2 ms; with textures (1600x1600 12 spp) 23.4 ->
// 18.5 ms, media (smoke box 400x400 64 spp) 7.8 -> 6.0 ms, a 160x120 4 spp
// preview 1.14 -> 0.67 ms.
//
// The grid is what stays resident (4 waves per SIMD); a wave leaves its loop
// when the shards are empty and its lanes' paths have ended, at most max_depth
// + 1 segments each.
#ifndef TPT_CSRC_PATHS_H
#define TPT_CSRC_PATHS_H

#include "render.h"

#pragma clang fp contract(off)

namespace tptd {

constexpr uint32_t PATH_THREADS = 256, PATH_WAVES = PATH_THREADS / 64;

// A wave's next up to 64 items (contiguous; *n of them), one atomic; 0 when the pass has none left.
__device__ __forceinline__ uint32_t claim_run(const pass_hdr &H, uint32_t *counters, uint32_t &shard, uint32_t *n) {
  for (uint32_t tries = 0; tries < NSUB; ++tries, shard = (shard + 1) % NSUB) {
    const uint32_t hi = shard_lo(H, shard + 1);
    uint32_t *cur = counters + cur_at(shard);
    if (__builtin_amdgcn_readfirstlane(__hip_atomic_load(cur, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) >= hi)
      continue;
    uint32_t base = 0;
    if (__lane_id() == 0) base = atomicAdd(cur, 64u);
    base = __builtin_amdgcn_readfirstlane(base);
    if (base >= hi) continue;
    *n = hi - base < 64u ? hi - base : 64u;
    return base;
  }
  *n = 0;
  return 0;
}

// SWEEP, SPH, MEDIA: the walk, as for k_trace; SIMPLE: the shading, as for k_shade.
// Waves per SIMD: 4 fit 128 VGPRs without spilling where one walk is compiled;
// the general walk needs 3 waves' registers, the general media walk 2.
__host__ __device__ constexpr uint32_t path_waves(bool sweep, bool sph, bool simple, bool media) {
  return sweep || sph || (simple && !media) ? 4u : (media ? 2u : 3u);
}

template <bool SWEEP, bool MULTI, bool SPH, bool SIMPLE, bool MEDIA = false>
__global__ void __launch_bounds__(PATH_THREADS) __attribute__((amdgpu_waves_per_eu(path_waves(SWEEP, SPH, SIMPLE, MEDIA))))
k_paths(scene_view S, const tpt_slot *__restrict__ slots, const tpt_entry *__restrict__ entries, render_params P,
        render_state Q) {
  S.slots = slots;
  S.entries = entries;
  // What the uniform pass knows of the hit, and the first draws of the shading: not in
  // the media variants, which have no registers left (smoke box 8% slower), and
  // not behind the tree walks (random spheres: 0.6% slower with the draws).
  constexpr bool kGeo = SWEEP && !MEDIA;
  const pass_hdr H = *P.hdr;
  // the wave's generated camera rays that no lane has taken yet: o, d, pixel, sample, entry
  __shared__ float pool[PATH_WAVES][9][64];
  __shared__ uint32_t bstack[SPH ? kBvhDepth * PATH_THREADS : 1];  // sphere_world's
  __shared__ unsigned long long acc[ST_BASIC];  // path_stats's
  if (threadIdx.x < ST_BASIC) acc[threadIdx.x] = 0;
  __syncthreads();
  const uint32_t wave = threadIdx.x / 64, lane = __lane_id();
  float(*mine)[64] = pool[wave];
  uint32_t pool_at = 0, pool_n = 0;  // wave-uniform
  bool more = true;
  uint32_t shard = (blockIdx.x * PATH_WAVES + wave) % NSUB;
  uint32_t st[ST_COUNT] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
  bool live = false;
  path p{};
  uint32_t px = 0, smp = 0;
  unsigned long long visits = 0;
  for (;;) {
    unsigned long long dead = __ballot(!live);
    while (dead != 0ull && (pool_n != 0u || more)) {
      if (pool_n == 0u) {
        uint32_t n;
        const uint32_t base = claim_run(H, Q.counters, shard, &n);
        if (n == 0u) {
          more = false;
          break;
        }
        if (lane < n) {
          const item_ctx c = item_in_entry(P, find_entry<MULTI>(P, H.n_ent, base + lane), base + lane);
          const path g = raygen(P, base + lane, c);
          mine[0][lane] = g.o.x, mine[1][lane] = g.o.y, mine[2][lane] = g.o.z;
          mine[3][lane] = g.d.x, mine[4][lane] = g.d.y, mine[5][lane] = g.d.z;
          mine[6][lane] = __uint_as_float(c.px), mine[7][lane] = __uint_as_float(c.smp);
          if (MULTI) mine[8][lane] = __uint_as_float(c.ent);
        }
        pool_at = 0;
        pool_n = n;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      }
      const uint32_t rank = lane_prefix(dead);
      const bool take = !live && rank < pool_n;
      if (take) {
        const uint32_t k = pool_at + rank;
        p.o = v3{mine[0][k], mine[1][k], mine[2][k]};
        p.d = v3{mine[3][k], mine[4][k], mine[5][k]};
        px = __float_as_uint(mine[6][k]), smp = __float_as_uint(mine[7][k]);
        if (MULTI) p.ent = __float_as_uint(mine[8][k]);
        p.thr = v3{1.0f, 1.0f, 1.0f};
        p.rad = v3{0.0f, 0.0f, 0.0f};
        p.depth = 0;
        live = true;
      }
      const uint32_t taken = __popcll(__ballot(take));
      pool_at += taken;
      pool_n -= taken;
      dead = __ballot(!live);
    }
    if (__ballot(live) == 0ull) break;
    const uint32_t job = MULTI ? P.pass[p.ent].job : 0u;
    const item_ctx c{p.ent, job, px, smp};
    const scene_view Sj = view_of<MULTI>(S, P, job);
    hit_t h{0.0f, kNone, kNone, 0};
    const ray_ctx rc = (MEDIA || (!SIMPLE && !SWEEP && !SPH)) && (P.motion | P.media) && live ? make_ray_ctx(P, c, p.depth)
                                                                                 : ray_ctx{0.0f, 0u, 0u, 0u, 0u, 0u};
    bool got;
    uint32_t nodes = 0;
    hit_geo geo{};
    if (SWEEP)
      got = small_world<false, MEDIA>(Sj, p.o, p.d, rc, 0.001f, kFltMax, &h, &nodes, live, nullptr,
                                      kGeo ? &geo : nullptr);
    else if (SPH)
      got = sphere_world<!MULTI, PATH_THREADS>(Sj, p.o, p.d, rc, 0.001f, kFltMax, live, bstack + threadIdx.x, &h,
                                               &nodes);
    else
      got = trace_world<false, MEDIA>(Sj, p.o, p.d, rc, 0.001f, kFltMax, &h, &nodes, live);
    if (!SWEEP) visits += nodes;
    if (live) {
      ++st[ST_SEGMENTS];
      uint32_t cls = Q_TERMINAL;
      if (got) {
        h.mat &= TPT_PAYLOAD_MASK;
        if (S.materials[h.mat].kind != TPT_MAT_DIFFUSE_LIGHT && p.depth < P.jobs[job].max_depth) cls = Q_OTHER;
      } else {
        h.slot = kNone;
      }
      if (!shade_hit<SIMPLE, MEDIA || !SIMPLE, kGeo>(S, Sj, P, P.jobs[job], c, p, h, cls, st,
                                                       kGeo ? &geo : nullptr)) {
        const pass_ent E = P.pass[MULTI ? p.ent : 0u];
        p.item = E.item_begin + (smp - E.s_begin) * P.jobs[job].n_pix + px;
        finish_sample<false>(P, Q, p, st);
        live = false;
      }
    }
  }
  path_stats(Q.stats, acc, st, visits, SWEEP ? S.n_flat : 0u);
}

}  // namespace tptd

#endif  // TPT_CSRC_PATHS_H
