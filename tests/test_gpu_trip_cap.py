"""What a ray that ends at the trip cap writes: the word of the node it is in
and its position."""
import numpy as np
import pytest

import svo_amd as S
from helpers import CONFIG1, params, path, scene_octree

pytestmark = pytest.mark.gpu


def test_word_and_position_at_the_cap():
    """The two rays of test_gpu_rays.test_trip_cap, whose y and z never become
    numbers again.  The values are the full rules' on the host, trip by trip
    for 2^22 trips in FP32, with the device's conversion of NaN to 0."""
    words, root = scene_octree(CONFIG1["kind"], CONFIG1["seed"], CONFIG1["depth"])
    p = params(CONFIG1, path(CONFIG1, 1), 0)
    for k in range(4):
        p.col0[k] = p.col1[k] = 0.0
    with S.Context(0) as c:
        c.upload_octree(words, root, 8)
        c.resize(16, 16)
        print("trip cap", flush=True)
        c.raycast_rect(p, 7, 7, 2, 1)
        c.sync()
        assert c.ray_stats() == (2, 1 << 22)
        assert c.screen(0)[7, 7:9].tolist() == [0xFF466C95] * 2
        xyz = np.ascontiguousarray(c.coords(0)[7, 7:9, :3])
        assert xyz[:, 0].view(np.uint32).tolist() == [1259489576] * 2
        assert np.isnan(xyz[:, 1]).all() and np.isneginf(xyz[:, 2]).all()
