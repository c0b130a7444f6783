"""Counts of a render that 32 bits do not hold, in a wave of one path launch.

Inside a perfect mirror ball every path goes to its depth limit, and a list of
thousands of rects outside it makes each segment count thousands of visits: 64
paths x 17601 segments x 4001 records = 4.5e9 in each of a block's four waves."""
import ctypes as C

import numpy as np
import pytest

import test_gpu_trace_lists as base

pytestmark = pytest.mark.gpu


def test_visits_of_a_wave_exceed_32_bits(tpt, device):
    rng = np.random.default_rng(1)
    far = [(2, 1, (y, x, x + 1.0, z, z + 1.0)) for x, y, z in rng.uniform(20, 30, (4000, 3))]
    sc, _ = base.scene(tpt, [[(1, 0, (0.0, 0.0, 0.0, -8.0))] + far], False, 0, False)  # (its normals point inwards)
    sc.close()
    mat = sc.host.keep[5]  # the same arrays with a metal of albedo 1 without fuzz
    mat[0] = 1
    for k in range(3):
        C.c_float.from_address(C.addressof(mat) + 8 + 4 * k).value = 1.0
    sc = tpt.Scene(sc.host)
    depth = 17600
    cam = tpt.camera_make((1.3, 0.2, 0.1), (1.0, 0.4, -2.0), (0.0, 1.0, 0.0), 60.0, 1.0, 0.0, 10.0)
    _, _, st = sc.render(width=16, height=16, spp=1, max_depth=depth, camera=cam, background=1.0)
    print(st["segments"], st["nodes_visited"], f"{st['kernel_ms']:.0f} ms", flush=True)
    assert st["paths"] == 256 and st["segments"] == 256 * (depth + 1)
    assert st["nodes_visited"] == st["segments"] * 4001
