"""svo_read_image_async into pinned memory: every alignment of the
destination, image sizes that are no multiple of 16 bytes, nothing written
beside the image; and the sets of the default pretrace when some images are
read and others are not."""
import numpy as np
import pytest

import svo_amd as S
from helpers import CONFIG1, assert_equal_u32, params, path, scene_octree

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def scene1():
    return scene_octree(CONFIG1["kind"], CONFIG1["seed"], CONFIG1["depth"])


@pytest.mark.parametrize("res", [(37, 21), (16, 16), (130, 67), (512, 256)])
@pytest.mark.parametrize("offset", [0, 1, 2, 3])
def test_copy_at_every_alignment(scene1, res, offset):
    words, root = scene1
    n, guard = res[0] * res[1], 0xA5A5A5A5
    c = S.Context(0)
    pin = S.PinnedImage(n + 64, 1)
    try:
        c.upload_octree(words, root, CONFIG1["depth"])
        c.resize(*res)
        c.frame_full(params(CONFIG1, path(CONFIG1, 2), 0))
        flat = pin.array.reshape(-1)
        flat[:] = guard
        o = 16 + offset
        pageable = np.zeros((res[1], res[0]), np.uint32)
        c.read_image_async(flat[o:o + n].reshape(res[1], res[0]))
        c.read_image_async(pageable)  # the same image again, another way
        c.sync()
        want = c.image().reshape(-1)
        assert_equal_u32(flat[o:o + n], want, "pinned")
        assert_equal_u32(pageable.reshape(-1), want, "pageable")
        assert np.all(flat[:o] == guard) and np.all(flat[o + n:] == guard)
        flat = None
    finally:
        pin.close()
        c.close()


@pytest.mark.parametrize("reads", [0b111111111111, 0b000111000111, 0b010101010101, 0b000000000001])
def test_frames_with_some_images_read(scene1, reads):
    """Frames issued ahead with the default pretrace, whose result sets go
    round by two after a frame that was read and by three after one that was
    not: images and screens equal frames without a pretrace."""
    words, root = scene1
    rx, ry = CONFIG1["res"]
    n = 12
    pr = path(CONFIG1, n)
    a, b = S.Context(0), S.Context(0)
    pins = [S.PinnedImage(rx, ry) for _ in range(n)]
    try:
        for c in (a, b):
            c.upload_octree(words, root, CONFIG1["depth"])
            c.resize(rx, ry)
        b.set_pretrace(sets=0)
        want = []
        for f in range(n):
            b.frame_warp(params(CONFIG1, pr, f))
            want.append(b.image())
        for f in range(n):
            a.frame_warp(params(CONFIG1, pr, f))
            if reads >> f & 1:
                a.read_image_async(pins[f].array)
        a.sync()
        for f in range(n):
            if reads >> f & 1:
                assert_equal_u32(pins[f].array, want[f], f"image {f}")
        assert_equal_u32(a.screen(), b.screen(), "screen planes")
        assert_equal_u32(a.image(), want[-1], "last image")
    finally:
        for p in pins:
            p.close()
        a.close()
        b.close()
