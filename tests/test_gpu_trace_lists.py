"""Small scenes with long lists in the uniform pass (walk_flat.h).

Scenes of at most 64 slots whose lists hold 11 boxes to 2400 rects, or hundreds of
spheres: around 64 primitives, around the 255 records of a class that one group
holds, under wrapper chains, and under a bvh.  The same scene with an empty
segment under a wrapper chain takes the general walk; leaf, t, record and
material must be the same bits.  The bounce loop's nodes_visited tells the route:
the pass counts every record once per segment."""
import ctypes as C
import struct
import types

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
PLAIN = 0x7FFFFFFF


class Entry(C.Structure):
    _fields_ = [("f", C.c_float * 5), ("xform", C.c_uint32), ("a", C.c_uint32), ("b", C.c_uint32)]


class Xform(C.Structure):
    _fields_ = [("nops", C.c_uint32), ("kinds", C.c_uint32), ("p", (C.c_float * 3) * 4), ("pad", C.c_uint32 * 2)]


def box6(lo, hi):
    (x0, y0, z0), (x1, y1, z1) = lo, hi
    return [(2, 2, (z1, x0, x1, y0, y1)), (2, 2, (z0, x0, x1, y0, y1)), (2, 1, (y1, x0, x1, z0, z1)),
            (2, 1, (y0, x0, x1, z0, z1)), (2, 0, (x1, y0, y1, z0, z1)), (2, 0, (x0, y0, y1, z0, z1))]


def lists_of(kind, rng):
    """Lists of (entry kind, axis, parameters), the records they make, and whether a bvh is over them."""
    def boxes(n):
        lo = rng.uniform(-12, 10, (n, 3))
        return [q for a, b in zip(lo, lo + rng.uniform(0.5, 2.5, (n, 3))) for q in box6(a, b)]

    def rects(n, axis=None):
        out = []
        for _ in range(n):
            k, a, b = rng.uniform(-12, 12, 3)
            out.append((2, int(rng.integers(3)) if axis is None else axis, (k, a, a + 1.0, b, b + 1.5)))
        return out

    def balls(n, r=0.4, at=None, wide=12.0):
        c = rng.uniform(-wide, wide, (n, 3)) + (0.0 if at is None else at)
        return [(1, 0, (*c[i], r)) for i in range(n)]

    if kind.startswith("boxes"):
        n = int(kind[5:])
        return [boxes(n)], n, False
    if kind.startswith("rects"):  # all of one axis
        n = int(kind[5:])
        return [rects(n, 1)], n, False
    if kind.startswith("balls"):
        n = int(kind[5:])
        return [balls(n)], n, False
    if kind == "mixed":
        return [boxes(40) + rects(100) + balls(70)], 210, False
    if kind == "lists":
        return [boxes(1) if k % 2 else rects(3) + balls(2) for k in range(32)], 16 + 16 * 5, True
    assert kind == "clusters"  # what path launches walk
    return [balls(16, 0.25, rng.uniform(-12, 12, 3), 0.8) for _ in range(32)], 512, True


def bounds(prims):
    lo, hi = np.full(3, np.inf), np.full(3, -np.inf)
    for kind, axis, p in prims:
        if kind == 1:
            a, b = np.array(p[:3]) - abs(p[3]), np.array(p[:3]) + abs(p[3])
        else:
            u, v = 1 if axis == 0 else 0, 1 if axis == 2 else 2
            a, b = np.zeros(3), np.zeros(3)
            a[axis], b[axis] = p[0] - 1e-3, p[0] + 1e-3
            a[u], b[u], a[v], b[v] = p[1], p[2], p[3], p[4]
        lo, hi = np.minimum(lo, a), np.maximum(hi, b)
    return lo, hi


def scene(tpt, lists, bvh, chains, general):
    slots, entries = [], []

    def leaf(k):
        slots.append(([struct.unpack("f", struct.pack("I", x))[0] for x in (len(entries), len(lists[k]))], len(entries),
                      (3 << 28) | len(entries)))
        for i, (kind, axis, p) in enumerate(lists[k]):
            entries.append((p, (len(entries) // 6) % chains if chains else 0xFFFFFFFF, axis << 28, kind))
        return bounds(lists[k])

    def build(ks, axis=0):
        if len(ks) == 1:
            return leaf(ks[0])
        ks = sorted(ks, key=lambda k: bounds(lists[k])[0][axis])
        at = len(slots)
        slots.append(None)
        a = build(ks[:len(ks) // 2], (axis + 1) % 3)
        right = len(slots)
        b = build(ks[len(ks) // 2:], (axis + 1) % 3)
        # (wide enough for the lists' float32 parameters)
        lo, hi = np.minimum(a[0], b[0]) - 1e-3, np.maximum(a[1], b[1]) + 1e-3
        slots[at] = ([*lo, *hi], len(slots), right)
        return lo, hi

    assert bvh or len(lists) == 1
    build(list(range(len(lists))))
    S, E = (tpt._Slot * len(slots))(), (Entry * len(entries))()
    for k, (f, a, b) in enumerate(slots):
        for i, x in enumerate(f):
            S[k].f[i] = x
        S[k].a, S[k].b = a, b
    for k, (f, x, a, b) in enumerate(entries):
        for i, y in enumerate(f):
            E[k].f[i] = y
        E[k].xform, E[k].a, E[k].b = x, a, b
    X = (Xform * (chains + 1))()  # the last: no operations
    for k in range(chains):
        X[k].nops, X[k].kinds = 2, 4  # translate, then rotate_y
        X[k].p[0][:] = [0.3 * k, -0.2 * k, 0.1]
        X[k].p[1][:] = [np.sin(0.2 * k + 0.1), np.cos(0.2 * k + 0.1), 0.0]
    segs = [0, len(slots)] + ([0, 0] if general else [])
    seg = (C.c_uint32 * len(segs))(*segs)
    wrap = (C.c_uint32 * 2)(PLAIN, chains)
    mat, tex = (C.c_uint32 * 8)(), (C.c_float * 8)(0, 0, 0, 0, 0.7, 0.6, 0.5)
    f = tpt.FlatScene()
    f.slots, f.n_slots, f.segments, f.n_segments = C.addressof(S), len(slots), C.addressof(seg), len(segs) // 2
    f.entries, f.n_entries, f.xforms, f.n_xforms = C.addressof(E), len(entries), C.addressof(X), chains + 1
    f.materials, f.n_materials, f.textures, f.n_textures = C.addressof(mat), 1, C.addressof(tex), 1
    f.n_leaves, f.max_depth = len(entries), 30
    if general:
        f.segment_xforms = C.addressof(wrap)
    f.bounds[:] = [-15.0] * 3 + [15.0] * 3
    info = types.SimpleNamespace(width=61, height=47, spp=2, max_depth=20, background=1.0)
    return tpt.Scene(types.SimpleNamespace(flat=f, keep=(S, E, X, seg, wrap, mat, tex), info=info)), len(entries)


KINDS = ["rects64", "rects65", "boxes10", "boxes11", "rects255", "rects256", "rects511", "balls64", "balls65", "balls300",
         "mixed", "boxes400", "lists", "clusters"]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("chains", [0, 3])
def test_long_lists(tpt, device, kind, chains):
    import torch

    if kind == "clusters" and chains:
        pytest.skip("wrapped spheres leave their boxes")
    rng = np.random.default_rng(len(kind) + chains)
    lists, records, bvh = lists_of(kind, rng)
    if bvh and chains:
        pytest.skip("wrapped lists leave their boxes")
    a, n = scene(tpt, lists, bvh, chains, False)
    b, _ = scene(tpt, lists, bvh, chains, True)
    # rays between points of the primitives, their corners among them
    prims = [q for q in sum(lists, [])]
    pts = []
    for ptype, axis, p in (prims[i] for i in rng.integers(0, len(prims), 1 << 16)):
        if ptype == 1:
            pts.append(p[:3])
        else:
            u, v = 1 if axis == 0 else 0, 1 if axis == 2 else 2
            x = np.zeros(3)
            x[axis] = p[0]
            x[u], x[v] = rng.choice([p[1], p[2], 0.5 * (p[1] + p[2])]), rng.choice([p[3], p[4], 0.5 * (p[3] + p[4])])
            pts.append(x)
    pts = np.array(pts)
    o = pts[rng.permutation(len(pts))] + rng.normal(size=pts.shape) * 10 ** rng.uniform(-5, 1, (len(pts), 1))
    d = pts + rng.normal(size=pts.shape) * 10 ** rng.uniform(-7, 0, (len(pts), 1)) - o
    d[::17, 0] = 0.0
    rays = torch.from_numpy(np.ascontiguousarray(np.concatenate([o, d], 1).T.astype(np.float32))).to(device)
    for tmin, tmax in ((0.001, 3.4028234663852886e38), (0.0, 0.7)):
        la, ta, ra, ma = a.trace(rays, tmin=tmin, tmax=tmax, record=True)
        lb, tb, rb, mb = b.trace(rays, tmin=tmin, tmax=tmax, record=True)
        assert torch.equal(la, lb)
        hit = lb >= 0
        assert float(hit.float().mean()) > 0.02
        assert torch.equal(ta[hit].view(torch.int32), tb[hit].view(torch.int32))
        assert torch.equal(ra[:, hit].view(torch.int32), rb[:, hit].view(torch.int32)) and torch.equal(ma, mb)
    # renders: the path launch, the bounce loop and the general walk give the same sums
    cam = tpt.camera_make((9.0, 7.0, 24.0), (0.0, 0.0, 0.0), (0.0, 1.0, 0.0), 60.0, 61 / 47, 0.0, 10.0)
    (sa, qa, st), (sl, ql, stl), (sb, qb, _) = [
        sc.render(camera=cam, seed=3, tail=tail) for sc, tail in ((a, True), (a, False), (b, True))]
    assert torch.equal(sa, sl) and torch.equal(qa, ql) and torch.equal(sa, sb) and torch.equal(qa, qb)
    assert stl["segments"] == st["segments"] > stl["paths"]
    if chains == 0:
        assert stl["nodes_visited"] == stl["segments"] * records  # the uniform pass
    else:
        assert stl["nodes_visited"] <= stl["segments"] * n and stl["nodes_visited"] % stl["segments"] == 0
    if kind == "clusters":
        assert st["nodes_visited"] < stl["nodes_visited"]  # walked
    elif chains == 0:
        assert st["nodes_visited"] == stl["nodes_visited"]
