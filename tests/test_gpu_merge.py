"""The merge of pretraced rays when a frame has more rays than the merge
launch has threads (its workgroups go round them), and when it has few."""
import numpy as np
import pytest

import svo_amd as S
from helpers import CONFIG1, assert_equal_u32, params, path, scene_octree

pytestmark = pytest.mark.gpu
THREADS = 512 * 256


@pytest.mark.parametrize("res", [(1920, 1024), (1361, 763), (64, 48)])
def test_merge_goes_round_all_rays(res):
    words, root = scene_octree(CONFIG1["kind"], CONFIG1["seed"], CONFIG1["depth"])
    pr = path(CONFIG1, 24)
    a, b = S.Context(0), S.Context(0)
    try:
        for c in (a, b):
            c.upload_octree(words, root, CONFIG1["depth"])
            c.resize(*res)
        a.set_pretrace(sets=3, only_queued=False)
        b.set_pretrace(sets=0)
        most = 0
        for i, f in enumerate((0, 1, 2, 3, 14, 15, 2, 23)):  # jumps: many holes
            p = params(CONFIG1, pr, f)
            p.frame = i
            for c in (a, b):
                c.frame_warp(p)
            a.sync()
            b.sync()
            assert_equal_u32(a.screen(), b.screen(), f"frame {i}")
            assert_equal_u32(a.image(), b.image(), f"frame {i} image")
            assert np.array_equal(a.coords(0).view(np.uint32), b.coords(0).view(np.uint32)), i
            rays = b.ray_stats(reset=True)[0]
            most = max(most, rays if i >= 2 else 0)
        merged = a.pretrace_stats()[1]
        assert merged > 0
        if res[0] == 1920:
            assert most > THREADS
    finally:
        a.close()
        b.close()
