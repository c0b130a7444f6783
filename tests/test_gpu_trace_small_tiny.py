"""Closest hits of small scenes along directions with a tiny component: from the
smallest denormal, whose reciprocal is infinite, through those whose reciprocal is
just finite, to ordinary ones, bit for bit with the oracle's walk."""
import numpy as np
import pytest

import test_gpu_trace_small as base

pytestmark = pytest.mark.gpu
TINY = [1e-45, 1e-40, 2.9e-39, 2.95e-39, 5e-39, 1.1e-38, 1.18e-38, 1e-37, 1e-30, 8e-19, 9e-19, 1e-18, 1e-10]


@pytest.mark.parametrize("name", base.SCENES)
def test_tiny_components_bit_exact(tpt, oracle, device, name):
    import torch

    s = oracle.scene(name)
    sc = tpt.Scene.named(name)
    rng = np.random.default_rng(3)
    # from points on the surfaces, where such a component decides about the plane it starts in
    for rays in (base.edge_rays(s, 1 << 15, 4), s.make_rays(1, 1 << 15, seed=5)):
        n = rays.shape[1]
        rays = rays.copy()
        leaf, t, rec, _ = s.trace(rays, record=True)
        on = (leaf >= 0) & np.isfinite(rec[2:5]).all(0) & (rng.random(n) < 0.7)
        rays[:3, on] = rec[2:5, on]
        cols, ax = np.arange(n), rng.integers(0, 3, n)
        rays[3 + ax, cols] = (rng.choice(TINY, n) * rng.choice([-1, 1], n)).astype(np.float32)
        two = rng.random(n) < 0.2
        rays[3 + (ax[two] + 1) % 3, cols[two]] = (rng.choice(TINY, two.sum())).astype(np.float32)
        for tmin, tmax in [(0.001, 3.4028234663852886e38), (0.0, 3e38), (-1.0, 2.0)]:
            want = s.trace(rays, tmin=tmin, tmax=tmax)
            got = [g.cpu().numpy() for g in sc.trace(torch.from_numpy(rays).to(device), tmin=tmin, tmax=tmax)]
            bad = np.nonzero(got[0] != want[0])[0]
            assert len(bad) == 0, (tmin, tmax, len(bad), rays[:, bad[:2]].T, got[0][bad[:2]], want[0][bad[:2]])
            hit = want[0] >= 0
            a, b = got[1][hit], want[1][hit]
            assert np.array_equal(np.isnan(a), np.isnan(b)), (tmin, tmax)
            ok = ~np.isnan(a)
            assert np.array_equal(a[ok].view(np.uint32), b[ok].view(np.uint32)), (tmin, tmax)
