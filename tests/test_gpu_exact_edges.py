"""Rays that cross cell edges exactly, vs the oracle bit-exact: directions of
power-of-two ratios from grid positions, so a step changes two axes at once.
Where one axis crosses the world's middle plane and another a quarter plane,
the XOR of the changes has bit D and no bit below it: not a pop, and no LOD
switch although one is due."""
import itertools

import numpy as np
import pytest

import oracle as O
import svo_amd as S
from helpers import assert_equal_f32_bits, assert_equal_u32

pytestmark = pytest.mark.gpu


def edge_slabs(depth):
    """Bars of 8x8 voxels along each axis behind the edges the rays cross."""
    n = 1 << (depth - 1)
    bars = []
    for a, b in itertools.permutations(range(3), 2):
        m = np.stack(np.meshgrid(np.arange(8), np.arange(n // 2, n // 2 + 8), np.arange(n), indexing="ij"), -1)
        v = np.empty((m.size // 3, 3), np.uint16)
        v[:, [a, b, 3 - a - b]] = m.reshape(-1, 3)
        bars.append(v)
    xyz = np.unique(np.concatenate(bars), axis=0)
    return S.build_octree(xyz, (np.arange(len(xyz), dtype=np.uint64) * 2654435761).astype(np.uint32), depth)


def edge_rays(depth, res, n):
    """(position, direction): axis a meets 2^depth in the step in which axis b
    meets 2^(depth-1) or three times that, after the first LOD switch is due."""
    rng = np.random.default_rng(100 * depth + res)
    for i in range(n):
        a, b = rng.permutation(3)[:2]
        k = int(rng.integers(res, 1 << (depth - 1)))
        pos, d = np.zeros(3), np.zeros(3)
        pos[a] = (1 << depth) - k
        pos[b] = int(rng.choice([1, 3])) * (1 << (depth - 1)) - k
        pos[3 - a - b] = rng.integers(0, 32 << depth) / 16.0
        d[[a, b]] = 1.0
        d[3 - a - b] = rng.choice([0.25, 0.5, 1.0])
        if rng.integers(2):  # another octant
            s = rng.integers(0, 2, 3) * 2 - 1
            pos, d = np.where(s < 0, (2 << depth) - pos, pos), d * s
        yield pos, d
    if depth == 8:
        yield np.array([156.0, 28.0, 10.0]), np.array([1.0, 1.0, 0.25])


def ray_params(pos, d):
    """A camera whose every pixel looks along d from pos (1/16 voxel units)."""
    p = S.FrameParams()
    for k in range(3):
        p.m0[k] = pos[k] / 16.0
        (p.col0, p.col1, p.col2)[k][2] = d[k]
    p.fovx = p.fovy = 1.0
    return p


@pytest.mark.parametrize("res", [16, 32, 64])
@pytest.mark.parametrize("depth", [8, 9, 11])
def test_middle_and_quarter_plane(depth, res):
    words, root = edge_slabs(depth)
    rays = [ray_params(*r) for r in edge_rays(depth, res, 240)]
    word = np.zeros(len(rays), np.uint32)
    xyz = np.zeros((len(rays), 3), np.float32)
    for i, p in enumerate(rays):
        word[i], xyz[i], _ = O.trace_pixel(words, root, depth, res, res, O.params_from(p), i % res, i // res)
    print(f"depth {depth} res {res}", flush=True)
    with S.Context(0) as c:
        c.upload_octree(words, root, depth)
        c.resize(res, res)
        for i, p in enumerate(rays):
            c.raycast_rect(p, i % res, i // res, 1, 1)
        c.sync()
        assert_equal_u32(c.screen(0).reshape(-1)[:len(rays)], word, "screen")
        assert_equal_f32_bits(c.coords(0).reshape(-1, 4)[:len(rays), :3], xyz, "coords")
