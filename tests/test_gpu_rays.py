"""The ray kernel's paths beside the common one, vs the oracle bit-exact:
octrees that share a normal record between depths (a node's kind then comes
from its block bits), every depth, rays that cross the world's middle planes
and edges many times or graze cell edges, and the trip cap."""
import numpy as np
import pytest

import oracle as O
import svo_amd as S
from helpers import CONFIG1, assert_equal_f32_bits, assert_equal_u32, params, path, scene_octree

pytestmark = pytest.mark.gpu


def shared_root(words, root):
    """The octree with one child of its root replaced by the root itself: the
    root's record is then reached at every depth, blocks at several."""
    w = words.copy()
    o = root >> 9
    j = next(j for j in range(8) if root >> j & 1)
    w[o + j] = (o << 9) | (root & 255)
    return w


def render(words, root, depth, p, res, **tuning):
    with S.Context(0) as c:
        c.upload_octree(words, root, depth)
        c.resize(*res)
        c.set_tuning(**tuning)
        c.frame_full(p)
        c.sync()
        return c.screen(0), c.coords(0)[..., :3], c.ray_stats()[1]


def oracle(words, root, depth, p, res):
    o = O.Frame(*res, words, root, depth, nthreads=8)
    o.frame_full(O.params_from(p))
    out = o.screen[0].copy(), o.coords[0][..., :3].copy()
    o.close()
    return out


@pytest.mark.parametrize("lds", [0, 512])
@pytest.mark.parametrize("f", [0, 5])
def test_shared_record_octree(f, lds):
    words, root = scene_octree(CONFIG1["kind"], CONFIG1["seed"], CONFIG1["depth"])
    w = shared_root(words, root)
    res = (177, 93)
    p = params(CONFIG1, path(CONFIG1, 6), f)
    print(f"shared record, frame {f}, lds {lds}", flush=True)
    scr, xyz, _ = render(w, root, 8, p, res, lds_cache_words=lds)
    ref = oracle(w, root, 8, p, res)
    assert not np.array_equal(ref[0], oracle(words, root, 8, p, res)[0])
    assert_equal_u32(scr, ref[0], "screen")
    assert_equal_f32_bits(xyz, ref[1], "coords")


@pytest.mark.parametrize("depth", [8, 9, 10, 13])
@pytest.mark.parametrize("view", ["level", "up", "diagonal", "corner"])
def test_sparse_world_crossings(depth, view):
    """A handful of voxels: most rays cross the repeated world until the far
    exit; axis-parallel and diagonal views meet cell edges and corners."""
    rng = np.random.default_rng(depth)
    n = 1 << depth
    xyz = rng.integers(0, n, (40, 3)).astype(np.uint16)
    words, root = S.build_octree(xyz, np.arange(1, 41, dtype=np.uint32) * 5, depth)
    yaw, pitch = {"level": (0.0, 0.0), "up": (0.3, -1.2), "diagonal": (np.pi / 4, 0.6154797), "corner": (2.1, 0.05)}[view]
    mid = n / 16.0  # the middle of the world (1 voxel = 1/8)
    pos = (mid, mid, mid) if view == "corner" else (mid + 3.3, mid - 2.7, mid + 1.9)
    p, _ = S.camera(yaw, pitch, 0.0, pos, depth, 0)
    res = (97, 61)
    print(f"depth {depth} {view}", flush=True)
    scr, xyz_out, _ = render(words, root, depth, p, res)
    ref = oracle(words, root, depth, p, res)
    assert_equal_u32(scr, ref[0], "screen")
    assert_equal_f32_bits(xyz_out, ref[1], "coords")


def test_trip_cap():
    """Two direction components of exactly zero leave a ray that never moves;
    it ends at the trip cap, wherever in a group of trips that falls."""
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


@pytest.mark.parametrize("wg", [1, 5])
@pytest.mark.parametrize("lanes", [1, 8, 64])
@pytest.mark.parametrize("group", [1, 64])
def test_hand_out(wg, lanes, group):
    """Each ray is handed out once, in launches with fewer waves of rays than
    the grid has, as many, and more (1 lane per wave): full frames (long
    blocks from the second on) and warp frames, ray counts included."""
    words, root = scene_octree(CONFIG1["kind"], CONFIG1["seed"], CONFIG1["depth"])
    rx, ry = 131, 67
    pr = path(CONFIG1, 5)
    o = O.Frame(rx, ry, words, root, 8, nthreads=8)
    with S.Context(0) as c:
        c.upload_octree(words, root, 8)
        c.resize(rx, ry)
        c.set_tuning(wg_per_cu=wg, refill=3, iters=16)
        c.set_ray_lanes(lanes)
        c.set_ray_spread(group, only_if_fits=False)
        c.set_long_first(300)
        c.set_pretrace(sets=0)
        for f in range(4):
            p = params(CONFIG1, pr, f)
            print(f"wg {wg} lanes {lanes} group {group} frame {f}", flush=True)
            c.ray_stats(reset=True)
            c.frame_warp(p)
            o.frame_warp(O.params_from(p))
            assert_equal_u32(c.screen(), o.screen, f"warp frame {f}")
            assert c.ray_count(reset=True) == c.hole_count() + rect_pixels(rx, ry, f)
        full = O.Frame(rx, ry, words, root, 8, nthreads=8)
        for f in range(2):
            p = params(CONFIG1, pr, f)
            c.ray_stats(reset=True)
            c.frame_full(p)
            full.frame_full(O.params_from(p))
            assert_equal_u32(c.screen(0), full.screen[0], f"full frame {f}")
            assert c.ray_count() == rx * ry
        full.close()
    o.close()


def rect_pixels(rx, ry, f):
    ax, ay, ex, ey = S.tile_schedule(rx, ry, f)
    return max(0, min(ax + ex, rx) - ax) * max(0, min(ay + ey, ry) - ay)


@pytest.mark.parametrize("n", [(1, 1), (8, 8), (9, 8), (64, 63), (131, 67)])
def test_rect_sizes(n):
    """Rectangles from one ray to the screen: pixels inside are the oracle's,
    the others keep the hole word, and each ray is counted once."""
    words, root = scene_octree(CONFIG1["kind"], CONFIG1["seed"], CONFIG1["depth"])
    rx, ry = 131, 67
    p = params(CONFIG1, path(CONFIG1, 1), 0)
    ref = oracle(words, root, 8, p, (rx, ry))[0]
    want = np.full((ry, rx), S.HOLE, np.uint32)
    want[:n[1], :n[0]] = ref[:n[1], :n[0]]
    with S.Context(0) as c:
        c.upload_octree(words, root, 8)
        c.resize(rx, ry)
        c.memset(0, S.HOLE, 4 * c.N)
        print(f"rect {n}", flush=True)
        c.raycast_rect(p, 0, 0, *n)
        assert_equal_u32(c.screen(0), want, "screen")
        assert c.ray_count() == n[0] * n[1]
