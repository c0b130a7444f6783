"""Closest hits of small scenes where rects lie in one plane, so that two are hit at
the same time: on a lattice of planes, with rays between lattice points, many of
them through edges; and where wrapped lists lie outside the boxes around them.
Bit for bit with the general walk (the same scene with an empty segment under a
wrapper chain)."""
import numpy as np
import pytest

import test_gpu_trace_lists as lists
import test_gpu_trace_spheres as base

pytestmark = pytest.mark.gpu


def lattice_rays(rng, n):
    o = np.round(rng.uniform(-10, 10, (n, 3)) * 2) / 2
    d = np.round(rng.uniform(-8, 8, (n, 3))) - o
    k = rng.integers(0, 6, n)
    ax, cols = rng.integers(0, 3, n), np.arange(n)
    d[cols[k == 0], ax[k == 0]] = 0.0
    d[cols[k == 1], ax[k == 1]] = rng.choice([1e-10, -1e-10, 1e-5], (k == 1).sum())
    d[k == 2] += rng.normal(size=((k == 2).sum(), 3)) * 10 ** rng.uniform(-9, -3, ((k == 2).sum(), 1))
    o[k == 3] += rng.normal(size=((k == 3).sum(), 3)) * 10 ** rng.uniform(-9, -3, ((k == 3).sum(), 1))
    d[(d == 0).all(1)] = 1.0
    return np.ascontiguousarray(np.concatenate([o, d], 1).T.astype(np.float32))


def rect_tree(rng, n):
    """n lattice rects, one slot each, under a bvh over their exact bounds."""
    rects = []
    for _ in range(n):
        k, a, b = np.round(rng.uniform(-8, 8, 3))
        rects.append((int(rng.integers(3)), (k, a, a + np.round(rng.uniform(1, 6)), b, b + np.round(rng.uniform(1, 6)))))
    out = []

    def build(ks, axis):
        if len(ks) == 1:
            i = ks[0]
            out.append((list(rects[i][1]) + [0.0], rects[i][0] << 28, (2 << 28) | i))
            return lists.bounds([(2, *rects[i])])
        at = len(out)
        out.append(None)
        ks = sorted(ks, key=lambda i: lists.bounds([(2, *rects[i])])[0][axis])
        a = build(ks[:len(ks) // 2], (axis + 1) % 3)
        right = len(out)
        b = build(ks[len(ks) // 2:], (axis + 1) % 3)
        # (whole numbers and their float32 neighbours: the plane's own 1e-3 is all the room there is)
        lo, hi = np.minimum(a[0], b[0]).astype(np.float32), np.maximum(a[1], b[1]).astype(np.float32)
        out[at] = (list(lo) + list(hi), len(out), right)
        return lo, hi

    build(list(range(n)), 0)
    return out, [(0, len(out))]


def compare(a, b, rays):
    import torch

    for tmin, tmax in ((0.001, 3.4028234663852886e38), (0.0, float("inf")), (-4.0, 2.0), (0.5, 1.0)):
        la, ta = a.trace(rays, tmin=tmin, tmax=tmax)
        lb, tb = b.trace(rays, tmin=tmin, tmax=tmax)
        bad = torch.nonzero(la != lb)[:2, 0].tolist()
        assert not bad, (tmin, tmax, [rays[:, i].tolist() for i in bad], la[bad].tolist(), lb[bad].tolist(), tb[bad].tolist())
        hit = (lb >= 0) & ~torch.isnan(tb)
        assert torch.equal(ta[hit].view(torch.int32), tb[hit].view(torch.int32)), (tmin, tmax)
    a.close()
    b.close()


@pytest.mark.parametrize("seed", range(12))
def test_coplanar_rects(tpt, device, seed):
    import torch

    rng = np.random.default_rng(seed)
    slots, segs = rect_tree(rng, int(rng.integers(6, 33)))
    rays = torch.from_numpy(lattice_rays(rng, 1 << 16)).to(device)
    compare(base.scene(tpt, slots, segs, 0), base.scene(tpt, slots, segs, 1), rays)


@pytest.mark.parametrize("seed", range(6))
@pytest.mark.parametrize("chains", [0, 1, 3])
def test_coplanar_boxes_in_lists(tpt, device, seed, chains):
    """Wrapped lists under a bvh lie outside the boxes around them (chains > 0)."""
    import torch

    rng = np.random.default_rng(100 + seed)
    parts = []
    for _ in range(int(rng.integers(2, 8))):
        lo = np.round(rng.uniform(-8, 4, (3, 3)))
        parts.append([q for a in lo for q in lists.box6(a, a + np.round(rng.uniform(1, 5, 3)))])
    a, _ = lists.scene(tpt, parts, True, chains, False)
    b, _ = lists.scene(tpt, parts, True, chains, True)
    compare(a, b, torch.from_numpy(lattice_rays(rng, 1 << 16)).to(device))
