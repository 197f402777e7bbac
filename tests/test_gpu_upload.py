"""svo_upload_octree's validation of many blocks: the block that is reported
is the first bad one in the order of the refs, whatever thread finds it, and
a bad block outranks a bad normal ref behind it."""
import numpy as np
import pytest

import svo_amd as S

pytestmark = pytest.mark.gpu
DEPTH = 10


@pytest.fixture(scope="module")
def octree():
    xyz, rgba = S.scene(2, 1002, DEPTH, 200)
    words, root = S.build_octree_gpu(xyz, rgba, DEPTH)
    # block refs in breadth-first order over the normal records
    blocks, queue = [], [root >> 9]
    for o in queue:
        for j in range(8):
            v = int(words[o + j])
            if v & 256:
                blocks.append(((v >> 9) << 6, o + j))
            elif v:
                queue.append(v >> 9)
    return words, root, blocks


def corrupt(words, base):
    """Clear the block bit of the block's first child ref; returns the node it names."""
    at = base + 1
    ref = int(words[at])
    assert ref & 256
    words[at] = ref & ~256
    return base + (ref >> 9)


@pytest.mark.parametrize("picks", [[0], [-1], [5, 70], [200, 90, 91], [63, 64, 65]])
def test_first_bad_block_is_reported(octree, picks):
    words, root, blocks = octree
    assert len(blocks) > 256  # several threads take part
    w = words.copy()
    named = {p % len(blocks): corrupt(w, blocks[p][0]) for p in picks}
    c = S.Context(0)
    try:
        for _ in range(5):
            with pytest.raises(S.SvoError) as e:
                c.upload_octree(w, root, DEPTH)
            assert f"(word {named[min(named)]})" in str(e.value)
        # a block ref behind them that lies in the normal region is an error of the walk: the block comes first
        w[blocks[-1][1]] = (w[blocks[-1][1]] & 0x1FF)
        if max(named) < len(blocks) - 1:
            with pytest.raises(S.SvoError) as e:
                c.upload_octree(w, root, DEPTH)
            assert f"(word {named[min(named)]})" in str(e.value)
        w = words.copy()
        w[blocks[-1][1]] &= 0x1FF
        with pytest.raises(S.SvoError) as e:
            c.upload_octree(w, root, DEPTH)
        assert "overlaps the normal region" in str(e.value)
        c.upload_octree(words, root, DEPTH)  # the untouched array is taken
    finally:
        c.close()


def test_words_live_as_long_as_their_views(octree):
    words, root, _ = octree
    a = words[100:200]
    b, _ = S.build_octree_gpu(np.array([[1, 2, 3]], np.uint16), np.array([7], np.uint32), 8)
    tail = b[-4:].copy()
    view = b[-4:]
    del b
    assert np.array_equal(view, tail) and a.base is not None
