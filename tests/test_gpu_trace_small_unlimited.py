"""Closest hits of small scenes without a limit: t_max = inf (and t_min = -inf),
bit for bit with the oracle's walk, at the cost of any other limit."""
import numpy as np
import pytest

import test_gpu_trace_small as base

pytestmark = pytest.mark.gpu
INF = float("inf")


@pytest.mark.parametrize("name", base.SCENES)
def test_unlimited_bit_exact(tpt, oracle, device, name):
    import torch

    s = oracle.scene(name)
    sc = tpt.Scene.named(name)
    special = base.special_rays(s, 1 << 15, 3)
    special[3:, ::9] = 0.0  # no direction at all
    special[3, ::18] = -0.0
    for rays in (base.edge_rays(s, 1 << 16, 4), special):
        for tmin, tmax in [(0.001, INF), (0.0, INF), (-INF, INF), (-INF, 3.0), (INF, INF), (-INF, -INF)]:
            want = s.trace(rays, tmin=tmin, tmax=tmax)
            got = [g.cpu().numpy() for g in sc.trace(torch.from_numpy(rays).to(device), tmin=tmin, tmax=tmax)]
            bad = np.nonzero(got[0] != want[0])[0]
            assert len(bad) == 0, (tmin, tmax, len(bad), rays[:, bad[:2]].T, got[0][bad[:2]], want[0][bad[:2]])
            hit = want[0] >= 0
            a, b = got[1][hit], want[1][hit]
            assert np.array_equal(np.isnan(a), np.isnan(b)), (tmin, tmax)
            ok = ~np.isnan(a)
            assert np.array_equal(a[ok].view(np.uint32), b[ok].view(np.uint32)), (tmin, tmax)


def test_unlimited_costs_no_more(tpt, oracle, device):
    """(With every ray undecided it took twice the time: 150 and 73 us for 2^21.)"""
    import torch

    sc = tpt.Scene.named("cornell555")
    rays = torch.from_numpy(oracle.scene("cornell555").make_rays(1, 1 << 21, seed=3)).to(device)

    def best(tmax):
        ms = []
        for _ in range(12):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            sc.trace(rays, tmax=tmax)
            b.record()
            b.synchronize()
            ms.append(a.elapsed_time(b))
        return min(ms)

    limited, unlimited = best(3e38), best(INF)
    print(f"2^21 rays: {limited * 1e3:.0f} us limited, {unlimited * 1e3:.0f} us not", flush=True)
    assert unlimited < 1.4 * limited
