"""Plain renders in one path launch per pass (k_paths) against the bounce loop.

By default a plain render carries every path through all its bounces in one
launch; with tail=False (TPT_RENDER_NO_TAIL) the bounce loop renders it.  The
scenes cover every variant of the kernel: each walk (small scenes, sphere-only,
general, media) with simple and with general shading, alone and pooled.  Same functions,
same Philox streams, samples summed in the same order: the sums must be equal
bit for bit and the counts the same, at sizes around a wave's 64 rays, the 64
work shards and a block's 256 threads.
"""
import pytest

pytestmark = pytest.mark.gpu

COUNTS = ("paths", "segments", "light_queries", "nodes_visited", "nan_samples")


@pytest.mark.parametrize("name", ["cornell555", "random_spheres", "random_spheres_n3000", "ref_cornell_box",
                                  "random_spheres_textured", "box_list", "cornell_smoke", "ref_random_scene"])
@pytest.mark.parametrize("w,h,spp,depth,offset", [
    (1, 1, 1, 50, 0),        # one path
    (9, 7, 1, 50, 3),        # 63 items: one short run of rays
    (13, 5, 1, 1, 0),        # 65 items, paths cut at depth 1
    (257, 1, 3, 0, 0),       # depth 0: every hit ends its path
    (61, 67, 5, 50, 2),      # ragged: 20435 items over 64 shards
    (320, 200, 9, 50, 1000),  # more items than lanes in flight
])
def test_paths_equal_bounce_loop(tpt, device, name, w, h, spp, depth, offset):
    import torch

    sc = tpt.Scene.named(name)
    i = sc.host.info
    cam = tpt.camera_make(tuple(i.lookfrom), tuple(i.lookat), (0.0, 1.0, 0.0), i.vfov, w / h, i.aperture, i.focus)
    kw = dict(width=w, height=h, spp=spp, seed=5, sample_offset=offset, max_depth=depth, camera=cam)
    a, qa, sa = sc.render(**kw)
    b, qb, sb = sc.render(tail=False, **kw)
    assert torch.equal(a, b) and torch.equal(qa, qb)
    for k in COUNTS:
        assert sa[k] == sb[k], k
    assert sa["paths"] == w * h * spp
    if name in ("cornell555", "random_spheres", "random_spheres_n3000"):  # the scenes that tail_* counts
        assert sa["tail_launches"] == 1 and sa["tail_segments"] == sa["segments"]
    assert sb["tail_launches"] == 0


POOLS = {
    "spheres": [f"random_spheres_n{n}" for n in (60, 900, 90, 2500, 300)],
    "textured spheres": ["random_spheres_textured", "random_spheres_n70", "random_spheres", "random_spheres_n400",
                         "random_spheres_textured"],
    "simple": ["cornell555", "random_spheres", "box_list", "cornell555", "random_spheres_n60"],
    "general": ["ref_cornell_box", "ref_random_scene", "ref_two_perlin_spheres", "box_list", "random_spheres"],
    "media": ["cornell_smoke", "ref_random_scene", "cornell555", "cornell_smoke", "random_spheres"],
}


@pytest.mark.parametrize("which", list(POOLS))
def test_paths_pooled_jobs_equal_bounce_loop(tpt, device, which):
    """Jobs of several scenes and sizes in one launch, sums without squares among them."""
    import torch

    hosts = [tpt.HostScene(n, seed=k + 1) for k, n in enumerate(POOLS[which])]
    pool = tpt.Scene.pool(hosts)

    def run(flags):
        jobs, bufs = [], []
        for k, (w, h, spp) in enumerate(((3, 1, 1), (64, 48, 5), (17, 33, 2), (80, 31, 3), (1, 65, 7))):
            j, s, q = pool.job(scene=k, width=w, height=h, spp=spp, seed=40 + k, max_depth=50,
                               sumsq_buf=False if k == 2 else None)
            jobs.append(j)
            bufs.append(s)
            if k != 2:
                bufs.append(q)
        L = tpt.Launch()
        L.flags = flags
        return bufs, pool.render_jobs(jobs, launch=L)

    (ba, sa), (bb, sb) = run(0), run(4)
    for x, y in zip(ba, bb):
        assert torch.equal(x, y)
    for k in COUNTS:
        assert sa[k] == sb[k], k
    assert sa["tail_launches"] == (1 if which == "spheres" else 0) and sb["tail_launches"] == 0


@pytest.mark.parametrize("name", ["cornell555", "ref_cornell_box", "random_spheres"])
@pytest.mark.parametrize("general", [False, True])
def test_pinhole_skips_the_lens_loop(tpt, device, name, general):
    """A zero lens without -0 coordinates skips the lens draws.

    Moving the camera from x = +0 to x = -0 takes the loop instead, and no value
    of a path depends on that sign: equal bits.
    """
    import torch

    sc = tpt.Scene.named(name)
    i = sc.host.info
    got = []
    for x in (0.0, -0.0):
        cam = tpt.camera_make((x, *tuple(i.lookfrom)[1:]), tuple(i.lookat), (0.0, 1.0, 0.0), i.vfov, 61 / 67, 0.0,
                              i.focus)
        got.append(sc.render(width=61, height=67, spp=5, seed=5, camera=cam, tail=not general))
    (a, qa, sa), (b, qb, sb) = got
    assert torch.equal(a, b) and torch.equal(qa, qb)
    assert all(sa[k] == sb[k] for k in COUNTS)
