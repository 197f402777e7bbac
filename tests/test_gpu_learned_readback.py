"""Learned frames with every image read while the next ones are issued: the
copies into pinned memory and the CNN share a stream, so each frame's CNN
queues behind the copy of the image before it."""
import numpy as np
import pytest

import svo_amd as S
from helpers import CONFIG1, assert_equal_u32, params, path, scene_octree
from svo_amd import learned

pytestmark = pytest.mark.gpu
FRAMES = 10


@pytest.mark.parametrize("fused", [True, False])
@pytest.mark.parametrize("way", ["pinned", "pageable", "both"])
def test_images_of_frames_issued_ahead(way, fused):
    words, root = scene_octree(CONFIG1["kind"], CONFIG1["seed"], CONFIG1["depth"])
    rx, ry = 261, 133
    flight = path(CONFIG1, FRAMES)
    cnn = S.Cnn(0)
    pins = [S.PinnedImage(rx, ry) for _ in range(FRAMES)]
    try:
        learned.load(cnn)
        cnn.set_fused(fused)
        with S.Context(0) as c:
            c.upload_octree(words, root, CONFIG1["depth"])
            c.resize(rx, ry)
            want = []
            for f in range(FRAMES):
                c.frame_warp_learned(cnn, params(CONFIG1, flight, f))
                want.append(c.image())
        assert any(not np.array_equal(a, b) for a, b in zip(want, want[1:]))
        pageable = [np.zeros((ry, rx), np.uint32) for _ in range(FRAMES)]
        with S.Context(0) as c:
            c.upload_octree(words, root, CONFIG1["depth"])
            c.resize(rx, ry)
            print(way, "fused" if fused else "per layer", flush=True)
            for f in range(FRAMES):
                c.frame_warp_learned(cnn, params(CONFIG1, flight, f))
                if way != "pageable":
                    c.read_image_async(pins[f].array)
                if way != "pinned":
                    c.read_image_async(pageable[f])
            c.sync()
        for f in range(FRAMES):
            if way != "pageable":
                assert_equal_u32(pins[f].array, want[f], f"frame {f}, pinned")
            if way != "pinned":
                assert_equal_u32(pageable[f], want[f], f"frame {f}, pageable")
    finally:
        cnn.close()
        for p in pins:
            p.close()
