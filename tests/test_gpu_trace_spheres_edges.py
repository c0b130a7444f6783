"""The tree of sphere-only scenes at the edges of what its builder accepts,
against the general walk as in test_gpu_trace_spheres: leaf and t the same bits."""
import numpy as np
import pytest

import test_gpu_trace_spheres as base

pytestmark = pytest.mark.gpu


def spheres(kind, rng):
    c, r = rng.uniform(-20, 20, (300, 3)), np.full(300, 0.3)
    if kind == "a denormal apart":  # no finite bin scale, whole or in part
        c[:100] = c[0]
        c[:100, 0] = 1e-39 * rng.integers(0, 9, 100)
    if kind == "all big":  # no sphere set aside: radii 2.5 to 9.9
        r = rng.uniform(2.5, 9.9, 300)
        c *= 4
    if kind == "big ones among big":  # 16 above 4 times the 17th, one as large as that
        r = rng.uniform(2.5, 4.0, 300)
        r[100], r[:16] = 16.0, np.linspace(64.5, 300.0, 16)
        r[8:16] *= -1
        r[101:] = np.minimum(r[101:], 3.9)
        c *= 10
    if kind == "one among big":
        r[:] = 2.5
        r[7] = 1000.0
        c *= 4
    return np.concatenate([c, r[:, None]], 1).astype(np.float32)


@pytest.mark.parametrize("kind", ["a denormal apart", "all big", "big ones among big", "one among big"])
@pytest.mark.parametrize("tree", [True, False])
def test_edges_equal_general_walk(tpt, device, kind, tree):
    import torch

    rng = np.random.default_rng(len(kind))
    s = spheres(kind, rng)
    slots, segs = base.slots_of(s, tree, rng)
    rays = torch.from_numpy(base.rays_for(s, rng, 1 << 17)).to(device)
    a = [x.cpu().numpy() for x in base.scene(tpt, slots, segs, False).trace(rays)]
    b = [x.cpu().numpy() for x in base.scene(tpt, slots, segs, True).trace(rays)]
    assert np.array_equal(a[0], b[0])
    hit = b[0] >= 0
    assert hit.mean() > 0.05
    assert np.array_equal(a[1][hit].view(np.uint32), b[1][hit].view(np.uint32))


def uneven(slots, how):
    """The trees of slots_of, one rule of theirs broken: a box high in the tree no
    longer holds what is below it, or does not name its second child."""
    slots = [(list(f), a, b) for f, a, b in slots]
    boxes = [i for i, x in enumerate(slots) if x[2] >> 28 == 0]
    if how == "cut":
        for i in boxes[:3]:
            f = slots[i][0]
            for k in range(3):
                f[3 + k] = 0.25 * f[k] + 0.75 * f[3 + k]
    else:
        for i in boxes[1:4]:
            slots[i] = (slots[i][0], slots[i][1], 0x0FFFFFFF)
    return slots


@pytest.mark.parametrize("how", ["cut", "one child"])
@pytest.mark.parametrize("n", [20, 300])  # the uniform pass, the tree
def test_uneven_boxes_are_walked_one_by_one(tpt, device, how, n):
    """A caller's boxes need not hold one another: what an outer box cuts off
    stays cut off."""
    import torch

    rng = np.random.default_rng(n)
    s = spheres("", rng)[:n]
    if n < 64:
        s[:, :3] *= 0.2
    slots, segs = base.slots_of(s, True, rng)
    slots = uneven(slots, how)
    rays = base.rays_for(s, rng, 1 << 16)
    rays[3, ::5] = 0.0  # undecided or general: what takes the exact paths
    rays[0, ::10] = s[0, 0]
    rays = torch.from_numpy(rays).to(device)
    a = [x.cpu().numpy() for x in base.scene(tpt, slots, segs, False).trace(rays)]
    b = [x.cpu().numpy() for x in base.scene(tpt, slots, segs, True).trace(rays)]
    assert np.array_equal(a[0], b[0])
    hit = b[0] >= 0
    assert hit.mean() > 0.01
    assert np.array_equal(a[1][hit].view(np.uint32), b[1][hit].view(np.uint32))
