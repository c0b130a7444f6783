"""The tree of sphere-only scenes (walk_bvh.h) against the general walk.

The same spheres with an empty segment under a wrapper chain are not traced as
sphere-only and take the general walk; leaf and t must be the same bits.  The scenes are what a
caller of the C ABI may hand over: one bvh segment, one segment per sphere (a
plain list), radii from 1e-3 to 50, hollow (negative) spheres, coincident ones
(equal t, the reference's order decides), equal centres, more big spheres than
the tree sets apart, coordinates that are not finite; and rays from inside,
from far away, grazing, with zero, tiny and NaN components.
"""
import ctypes as C
import types

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def spheres(kind, rng):
    n = {"bvh": 700, "list": 150, "radii": 400, "many big": 200, "ties": 300, "one": 65, "nan": 120}[kind]
    c = rng.uniform(-20, 20, (n, 3))
    c[:, 1] *= 0.2
    r = np.full(n, 0.3)
    if kind == "radii":
        r = 10 ** rng.uniform(-3, 0.2, n)
        r[:3] = [50.0, 30.0, -12.0]
        r[10:40] *= -1
    if kind == "many big":
        r[:40] = rng.uniform(2.5, 6.0, 40)
    if kind == "ties":
        c[100:200] = c[0:100]  # coincident pairs
        r[100:150] *= -1
        c[200:] = c[200]  # equal centres, nested
        r[200:] = np.linspace(0.1, 1.5, 100)
    if kind == "one":
        c[:] = c[0]
        r[:] = 0.5  # every sphere the same
    if kind == "nan":
        c[7, 1] = np.nan
        c[9, 0] = np.inf
    return np.concatenate([c, r[:, None]], 1).astype(np.float32)


def slots_of(s, tree, rng):
    """Slots and segments: one bvh over all spheres (boxes exact unions, random
    axes, as the reference's bvh_node builds them), or one segment each."""
    out = []

    def leaf(i):
        f = list(s[i]) + [0.0, 0.0]
        out.append((f, 0, (1 << 28) | i))

    if not tree:
        for i in range(len(s)):
            leaf(i)
        return out, [(i, i + 1) for i in range(len(s))]
    order = {}

    def build(idx):
        at = len(out)
        out.append(None)
        if len(idx) > 2:
            idx = idx[np.argsort(s[idx, rng.integers(0, 3)], kind="stable")]
        half = len(idx) // 2
        parts = [idx[:half], idx[half:]] if len(idx) > 1 else [idx]
        boxes, right = [], 0x0FFFFFFF
        for k, p in enumerate(parts):
            if k:
                right = len(out)
            if len(p) == 1:
                i = int(p[0])
                order[len(order)] = i
                leaf(i)
                rr = s[i, 3]
                boxes.append((s[i, :3] - rr, s[i, :3] + rr))
            else:
                boxes.append(build(p))
        lo = np.minimum.reduce([b[0] for b in boxes])
        hi = np.maximum.reduce([b[1] for b in boxes])
        out[at] = (list(lo) + list(hi), len(out), right)
        return lo, hi

    build(np.arange(len(s)))
    return out, [(0, len(out))]


def scene(tpt, slots, segs, general):
    slots, segs = list(slots), list(segs)
    n_leaves = sum(1 for x in slots if x[2] >> 28)
    if general:
        segs.append((0, 0))
    f = tpt.FlatScene()
    arr = (tpt._Slot * len(slots))()
    for k, (v, a, b) in enumerate(slots):
        arr[k].f[:] = [float(x) for x in v]
        arr[k].a, arr[k].b = a, b
    seg = (C.c_uint32 * (2 * len(segs)))(*[x for s in segs for x in s])
    mat = (C.c_uint32 * 8)()  # one lambertian with texture 0
    tex = (C.c_uint32 * 8)()
    f.slots, f.n_slots = C.addressof(arr), len(slots)
    f.segments, f.n_segments = C.addressof(seg), len(segs)
    f.materials, f.n_materials = C.addressof(mat), 1
    f.textures, f.n_textures = C.addressof(tex), 1
    f.n_leaves, f.max_depth = n_leaves, 30
    wrap = (C.c_uint32 * len(segs))(*([0x7FFFFFFF] * (len(segs) - 1) + [0 if general else 0x7FFFFFFF]))
    xf = (C.c_uint32 * 16)()  # a chain of no operations
    f.segment_xforms = C.addressof(wrap)
    f.xforms, f.n_xforms = C.addressof(xf), 1
    f.bounds[:] = [-25.0] * 3 + [25.0] * 3
    return tpt.Scene(types.SimpleNamespace(flat=f, keep=(arr, seg, mat, tex, wrap, xf)))


def rays_for(s, rng, n):
    ok = s[np.isfinite(s).all(1)]
    q = rng.integers(0, len(ok), n)
    c, r = ok[q, :3].astype(np.float64), np.abs(ok[q, 3]).astype(np.float64)
    u = rng.normal(size=(n, 3))
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    kind = rng.integers(0, 7, n)
    o = rng.uniform(-25, 25, (n, 3))
    far = kind == 1
    o[far] = u[far] * 10 ** rng.uniform(1.5, 4.5, (far.sum(), 1))
    sur = kind == 2  # on a surface
    o[sur] = c[sur] + u[sur] * r[sur, None]
    ins = kind == 3
    o[ins] = c[ins] + u[ins] * r[ins, None] * rng.uniform(0, 1, (ins.sum(), 1))
    w = rng.normal(size=(n, 3))
    w -= (w * u).sum(1, keepdims=True) * u
    w /= np.linalg.norm(w, axis=1, keepdims=True)
    tgt = c + w * r[:, None] * (1 + rng.choice([-1, 1, 0], n) * 10 ** rng.uniform(-7, -1, n))[:, None]
    d = tgt - o
    d[ins] = rng.normal(size=(ins.sum(), 3))
    d /= np.maximum(np.linalg.norm(d, axis=1, keepdims=True), 1e-12)
    d *= 2.0 ** rng.integers(-5, 6, (n, 1))
    ax = rng.integers(0, 3, n)
    z = kind == 4
    d[z, ax[z]] = 0.0
    z = kind == 5
    d[z, ax[z]] *= 10 ** rng.uniform(-20, -2, z.sum())
    out = np.concatenate([o, d], 1).astype(np.float32)
    out[:20, 0] = np.nan
    out[20:40, 4] = np.nan
    out[40:60, 3:] = 0.0
    out[60:80, 3:] *= np.float32(1e-25)
    return np.ascontiguousarray(out.T)


@pytest.mark.parametrize("kind", ["bvh", "list", "radii", "many big", "ties", "one", "nan"])
@pytest.mark.parametrize("tree", [True, False])
def test_sphere_tree_equals_general_walk(tpt, device, kind, tree):
    import torch

    rng = np.random.default_rng(len(kind) * 7 + tree)
    s = spheres(kind, rng)
    if tree and kind == "nan":
        s[~np.isfinite(s)] = 3e38  # a box of infinite size instead
    slots, segs = slots_of(s, tree, rng)
    a, b = scene(tpt, slots, segs, 0), scene(tpt, slots, segs, 1)
    rays = torch.from_numpy(rays_for(s, rng, 1 << 16)).to(device)
    for tmin, tmax in [(0.001, 3.4028234663852886e38), (0.0, 12.0), (-3.0, 3e38), (2.0, 9.0), (4.0, 1.0)]:
        la, ta = a.trace(rays, tmin=tmin, tmax=tmax)
        lb, tb = b.trace(rays, tmin=tmin, tmax=tmax)
        bad = torch.nonzero(la != lb)[:3, 0].tolist()
        assert not bad, (tmin, tmax, [rays[:, i].tolist() for i in bad], la[bad].tolist(), lb[bad].tolist())
        hit = la >= 0
        assert torch.equal(ta[hit].view(torch.int32), tb[hit].view(torch.int32)), (tmin, tmax)
        print(kind, tree, tmin, tmax, f"hit {float(hit.float().mean()):.3f}", flush=True)
    a.close()
    b.close()
