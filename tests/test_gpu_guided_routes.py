"""Which route a guided render takes, told by its statistics, and a guided render
of media in the uniform pass against the general walk."""
import ctypes as C
import types

import pytest

pytestmark = pytest.mark.gpu


def render(tpt, sc, i, w, h, spp, **kw):
    cam = tpt.camera_make(tuple(i.lookfrom), tuple(i.lookat), (0.0, 1.0, 0.0), i.vfov, w / h, i.aperture, i.focus)
    g = tpt.Guide(seed=9)
    s, q, st = sc.render(width=w, height=h, spp=spp, seed=5, camera=cam, max_depth=50, guide=g, profile=True, **kw)
    return s, q, st, g


@pytest.mark.parametrize("name", ["cornell555", "random_spheres"])
@pytest.mark.parametrize("verts,cap,direct", [(1, 0, True), (2, 0, True), (4, 0, True), (5, 0, False),
                                              (1, 1 << 12, False), (4, 1 << 12, False)])
def test_the_tail_follows_the_guided_vertices(tpt, device, name, verts, cap, direct):
    """Every path in flight from the start (28609 items; not with 4096 records) and
    at most 4 guided vertices: one bounce per guided vertex, then the tail, and again
    after each shading of handed-back vertices.  Else the bounces go on until few
    paths are left."""
    sc = tpt.Scene.named(name)
    _, _, st, _ = render(tpt, sc, sc.host.info, 67, 61, 7, guide_vertices=verts, guiding=4, queue_capacity=cap)
    share = st["tail_segments"] / st["segments"]
    print(name, verts, cap, st["trace_launches"], st["tail_launches"], f"{share:.3f}", flush=True)
    if direct:
        assert st["trace_launches"] == verts and st["tail_launches"] >= 2 and share > 0.05
    else:
        assert st["trace_launches"] >= 8 and share < 0.05


def test_guided_media_in_the_uniform_pass(tpt, device):
    """The smoke box with an empty segment under a wrapper chain takes the general
    media walk: the same sums, squares and recorded rows, bit for bit."""
    import torch

    host = tpt.HostScene("cornell_smoke")
    f = tpt.FlatScene.from_buffer_copy(host.flat)
    n = f.n_segments
    old = (C.c_uint32 * (2 * n)).from_address(f.segments)
    seg = (C.c_uint32 * (2 * n + 2))(*old, 0, 0)
    wrap = (C.c_uint32 * (n + 1))(*[0x7FFFFFFF] * n, 0)
    assert f.n_xforms > 0 and not f.segment_xforms
    f.segments, f.n_segments, f.segment_xforms = C.addressof(seg), n + 1, C.addressof(wrap)
    general = tpt.Scene(types.SimpleNamespace(flat=f, keep=(host, seg, wrap), info=host.info, camera=host.camera))
    for verts in (2, 6):
        for scatter in (False, True):
            kw = dict(guide_vertices=verts, guiding=4, media_scatter=scatter)
            a, qa, sa, ga = render(tpt, tpt.Scene(host), host.info, 67, 61, 7, **kw)
            b, qb, sb, gb = render(tpt, general, host.info, 67, 61, 7, **kw)
            assert torch.equal(a, b) and torch.equal(qa, qb) and torch.equal(ga.copy_rows(), gb.copy_rows())
            assert sa["segments"] == sb["segments"]
            # the pass counts each record in every segment: a box or medium is one
            assert sa["nodes_visited"] % sa["segments"] == 0 and sa["nodes_visited"] != sb["nodes_visited"]
