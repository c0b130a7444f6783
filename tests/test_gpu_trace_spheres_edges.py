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
    return np.concatenate([c, r[:, None]], 1).astype(np.float32)


@pytest.mark.parametrize("kind", ["a denormal apart"])
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
