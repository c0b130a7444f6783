"""Closest hits of small scenes where the uniform pass (walk_flat.h) decides by
error bounds: rays aimed at edges and corners of rects and boxes, rays starting
on surfaces and next to edges, zero direction components (in-plane rays hit at
t = NaN), NaN origins, and t_min / t_max next to the hit, all bit for bit with
the oracle's walk."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SCENES = ["cornell555", "ref_cornell_box", "ref_sphere_cornell_box", "ref_light_spheres", "ref_two_perlin_spheres",
          "cornell_smoke"]


def unit(v):
    return v / np.linalg.norm(v, axis=1, keepdims=True)


def edge_rays(s, n, seed):
    """Rays from random surface points toward points next to other hits' edges:
    a hit's coordinates snapped to the scene's own plane coordinates (1 to 3 of
    them), moved off by 0 to 1e-2."""
    rng = np.random.default_rng(seed)
    base = np.concatenate([s.make_rays(0, n // 2, seed=seed), s.make_rays(1, n - n // 2, seed=seed + 1)], axis=1)
    leaf, t, rec, mat = s.trace(base, record=True)
    p = rec[2:5].T.astype(np.float64)
    hit = (leaf >= 0) & np.isfinite(p).all(1)
    p = p[hit]
    # coordinates that many hits share are the planes of the walls and boxes
    planes = []
    for c in range(3):
        v, k = np.unique(np.round(p[:, c], 2), return_counts=True)
        planes.append(v[np.argsort(-k)[:8]])
    m = n
    o = p[rng.integers(0, len(p), m)]
    q = p[rng.integers(0, len(p), m)].copy()
    for c in range(3):
        snap = rng.random(m) < 0.6
        q[snap, c] = planes[c][rng.integers(0, len(planes[c]), snap.sum())]
    q += rng.choice([-1, 0, 1], (m, 3)) * 10 ** rng.uniform(-7, -2, (m, 3))
    o += rng.choice([0, 0, 1], (m, 3)) * rng.normal(size=(m, 3)) * 10 ** rng.uniform(-6, -1, (m, 1))
    d = q - o
    d[np.linalg.norm(d, axis=1) == 0] = 1.0
    d = unit(d) * 2.0 ** rng.integers(-4, 9, (m, 1))
    return np.ascontiguousarray(np.concatenate([o, d], 1).T.astype(np.float32))


def special_rays(s, n, seed):
    """One or two zero direction components, grazing directions from surfaces,
    NaN and partly NaN origins, tiny and huge components."""
    rng = np.random.default_rng(seed)
    r = s.make_rays(1, n, seed=seed).copy()
    k = rng.integers(0, 7, n)
    ax = rng.integers(0, 3, n)
    cols = np.arange(n)
    r[3 + ax[k == 0], cols[k == 0]] = 0.0
    m = k == 1  # along one axis, as the reference's lights without a sampler send them
    r[3:, m] = 0.0
    r[3 + ax[m], cols[m]] = rng.choice([-1.0, 1.0], m.sum())
    m = k == 2
    r[3 + ax[m], cols[m]] *= np.float32(10.0) ** rng.uniform(-12, -3, m.sum()).astype(np.float32)
    r[:3, k == 3] = np.nan
    m = k == 4
    r[ax[m], cols[m]] = np.nan
    m = k == 5
    r[3 + ax[m], cols[m]] = rng.choice([1e-30, -1e-30, 1e25, np.nan, -0.0], m.sum())
    return r


@pytest.mark.parametrize("name", SCENES)
def test_small_scene_edges_bit_exact(tpt, oracle, device, name):
    import torch

    s = oracle.scene(name)
    sc = tpt.Scene.named(name)
    sets = {"edges": edge_rays(s, 1 << 17, 5), "special": special_rays(s, 1 << 16, 9)}
    for what, rays in sets.items():
        leaf, t = s.trace(rays)
        near = float(np.median(t[(leaf >= 0) & np.isfinite(t)]))
        for tmin, tmax in [(0.001, 3.4028234663852886e38), (0.0, 3e38), (-1.0, near), (near, 2 * near), (5.0, 1.0)]:
            want = s.trace(rays, tmin=tmin, tmax=tmax)
            got = [g.cpu().numpy() for g in sc.trace(torch.from_numpy(rays).to(device), tmin=tmin, tmax=tmax)]
            bad = np.nonzero(got[0] != want[0])[0]
            assert len(bad) == 0, (what, tmin, tmax, len(bad), rays[:, bad[:2]].T, got[0][bad[:2]], want[0][bad[:2]])
            hit = want[0] >= 0
            a, b = got[1][hit], want[1][hit]
            assert np.array_equal(np.isnan(a), np.isnan(b)), (what, tmin, tmax)
            ok = ~np.isnan(a)
            assert np.array_equal(a[ok].view(np.uint32), b[ok].view(np.uint32)), (what, tmin, tmax)
            print(name, what, tmin, tmax, f"hit {hit.mean():.3f} nan {np.isnan(b).sum()}", flush=True)
