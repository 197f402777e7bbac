"""The gate's ballot of 2x2 quads and its copy of plane 0 at sizes with cut
tiles and blocks, against the oracle's gated frame; the ray ranges of a batch
of more views than a wave has lanes."""
import numpy as np
import pytest

import oracle as O
import svo_amd as S
from svo_amd import workloads as W
from helpers import assert_equal_f32_bits, assert_equal_u32

pytestmark = pytest.mark.gpu
NAME = "flythrough_256"


@pytest.mark.parametrize("res", [(16, 16), (37, 21), (33, 48), (130, 67), (257, 129)])
@pytest.mark.parametrize("max_holes,max_depth", [(0, 0.0), (3, 60.0), (64, 0.0)])
def test_gate_at_odd_sizes(res, max_holes, max_depth):
    words, root, depth, _ = W.octree(NAME)
    rows = W.path(NAME, 8)
    o = O.Frame(res[0], res[1], words, root, depth, nthreads=8)
    with S.Context(0) as c:
        c.upload_octree(words, root, depth)
        c.resize(*res)
        c.set_gate_depth(max_depth)
        for f in range(8):
            p = W.frame_params(NAME, rows, f)
            c.frame_warp_learned(None, p, max_holes)
            o.frame_warp_gated(O.params_from(p), max_holes, max_depth)
            c.sync()
            assert_equal_u32(c.screen(), o.screen, f"frame {f} screen")
            assert_equal_f32_bits(c.coords(), o.coords, f"frame {f} coords")
            assert_equal_u32(c.image(), o.image, f"frame {f} image")
    o.close()


def test_batch_of_more_views_than_lanes():
    words, root, depth, _ = W.octree(NAME)
    rows = W.path(NAME, 4)
    n = 66
    sizes = [(16 + 8 * (i % 5), 16 + 16 * (i % 3)) for i in range(n)]
    views = [S.Context(0) for _ in range(n)]
    one = S.Context(0)
    try:
        for c, r in zip(views, sizes):
            c.upload_octree(words, root, depth)
            c.resize(*r)
        b = S.Batch(views)
        for f in range(4):
            b.frame_warp_learned(None, [W.frame_params(NAME, rows, f) for _ in range(n)])
        b.sync()
        one.upload_octree(words, root, depth)
        for i in (0, 1, 63, 64, 65):
            one.resize(*sizes[i])
            for f in range(4):
                one.frame_warp_learned(None, W.frame_params(NAME, rows, f))
            one.sync()
            assert_equal_u32(views[i].screen(), one.screen(), f"view {i}")
            assert_equal_u32(views[i].image(), one.image(), f"view {i} image")
        b.close()
    finally:
        one.close()
        for c in views:
            c.close()
