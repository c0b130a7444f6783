"""Guided renders whose tail follows the guided vertices directly.

That route is taken where every path is in flight from the start and at most 4
vertices are guided; its waves refill ended lanes, and it repeats after each
shading of handed-back vertices.  Same functions, same Philox streams: sums,
counts and recorded rows equal the bounce loop's (tail=False) bit for bit, on
both sides of each limit, from one path to more than the lanes in flight.
"""
import pytest

pytestmark = pytest.mark.gpu

COUNTS = ("paths", "segments", "light_queries", "nodes_visited", "nan_samples")


@pytest.mark.parametrize("name", ["cornell555", "random_spheres"])
@pytest.mark.parametrize("verts", [1, 2, 4, 5])
@pytest.mark.parametrize("w,h,spp,depth,cap", [
    (1, 1, 1, 50, 0),           # one path
    (13, 5, 1, 1, 0),           # 65 paths cut at depth 1
    (67, 61, 7, 50, 0),         # ragged, all in flight
    (67, 61, 7, 50, 1 << 12),   # more items than records: the polled route
    (320, 200, 9, 50, 0),       # more records than the tail's lanes
])
def test_guided_tail_equals_bounce_loop(tpt, device, name, verts, w, h, spp, depth, cap):
    import torch

    sc = tpt.Scene.named(name)
    i = sc.host.info
    cam = tpt.camera_make(tuple(i.lookfrom), tuple(i.lookat), (0.0, 1.0, 0.0), i.vfov, w / h, i.aperture, i.focus)
    g = tpt.Guide(seed=9)
    kw = dict(width=w, height=h, spp=spp, seed=5, camera=cam, max_depth=depth, queue_capacity=cap, guide=g,
              guide_vertices=verts, guiding=4)
    a, qa, sa = sc.render(**kw)
    rows = g.copy_rows()
    b, qb, sb = sc.render(tail=False, **kw)
    assert torch.equal(a, b) and torch.equal(qa, qb) and torch.equal(rows, g.copy_rows())
    assert all(sa[k] == sb[k] for k in COUNTS)
    assert sa["paths"] == w * h * spp and sb["tail_launches"] == 0
