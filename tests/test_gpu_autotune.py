"""tpt_autotune where the settings make no difference, and where a flag makes it.

Plain jobs take one path launch per pass whatever the settings, so the tuner has
nothing to choose: it must not return whichever of nine equal trials noise made
the fastest, nor spend their time.  With TPT_RENDER_NO_TAIL they run the bounce
loop, and that is what the trials must time."""
import time

import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def pool(tpt, device):
    return tpt.Scene.pool([tpt.HostScene(f"random_spheres_n{n}", seed=n) for n in (300, 900, 2000)])


def jobs_of(pool):
    out = [pool.job(scene=k, width=320, height=200, spp=64, seed=k, max_depth=20) for k in range(3)]
    return [j for j, _, _ in out], [b for _, s, q in out for b in (s, q)]


def test_plain_jobs_are_timed_once(tpt, pool):
    jobs, _ = jobs_of(pool)
    caps, _ = tpt.autotune_plan(jobs, calib_spp=1)
    for _ in range(6):
        best, ms = pool.autotune(jobs, calib_spp=1)
        assert (best.queue_capacity, best.blocks_per_cu, best.graph_iters) == (caps[-1], 64, 0)
        assert ms > 0


def test_the_bounce_loop_is_tuned_as_it_runs(tpt, pool):
    import torch

    jobs, _ = jobs_of(pool)
    caps, _ = tpt.autotune_plan(jobs, calib_spp=1)
    L = tpt.Launch()
    L.flags = 4
    t0 = time.perf_counter()
    plain, plain_ms = pool.autotune(jobs, calib_spp=1)
    t1 = time.perf_counter()
    best, ms = pool.autotune(jobs, calib_spp=1, base=L)
    t2 = time.perf_counter()
    assert best.flags == 4 and best.queue_capacity in caps and best.blocks_per_cu in (16, 32, 64)
    print(f"plain {plain_ms:.2f} ms in {t1 - t0:.3f} s, bounce loop {ms:.2f} ms in {t2 - t1:.3f} s", flush=True)
    assert ms > 1.2 * plain_ms  # (the loop takes two to three times as long)
    (ja, a), (jb, b) = jobs_of(pool), jobs_of(pool)
    pool.render_jobs(ja, launch=best)
    pool.render_jobs(jb)
    assert all(torch.equal(x, y) for x, y in zip(a, b))
