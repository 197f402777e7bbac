"""Timed cases of the framework: what a program that renders, trains or loads
scenes with it does, through the public binding (svo_amd).

A case is a dict of plain values; its "path" names the program:

  clip    a camera flight: `frames` successive frames of one context, each
          frame's image copied into pinned host memory as a headless renderer
          or an encoder feed does (mode "warp", "learned" or "full")
  still   an interactive viewer: one warp frame, its image read back blocking
  stages  the reference's own host loop (memset, proj, compaction, hole rays,
          tile refresh, copy, fill, colorize), one library call per kernel
  batch   many cameras of one scene with the learned fill, as a server runs
          them: one batch frame, every view's image read back
  proj    the warp alone on the caller's device buffers
  train   the hole filler's training loop: pair rendering and Adam steps,
          then the parameters as a checkpoint takes them
  grads   loss and gradients of a crop batch from host memory
  scene   a scene edit: build the octree of a voxel stream, upload it, show it

Scenes: kind 1 is the two-octave heightfield, kind 2 the fractal terrain with
spheres, kind 4 the 3-D noise cave; sizes follow the repository's workloads
(512x256 at depth 8, 1920x1024 at depth 11, the views' resolutions) and the
steps between them.  The seed chooses the camera flight (and the voxels or
tensors where those are the input); a scene is an asset that programs share.
"""
import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "sparse-voxel-octree-raycasting_amd"))

import svo_amd as S  # noqa: E402
from svo_amd import learned  # noqa: E402

DEPTHS = {1: (8, 9), 2: (9, 10, 11), 4: (8, 9, 10)}  # scene kinds and the depths they are used at
VIEWS = ((320, 240), (640, 480), (1280, 720), (1920, 1024))
PATH_FRAMES = 64  # length of a flight; it is flown back and forth
WARM_FRAMES = 6   # frames rendered before the timed ones: the caches hold a real frame


def listed():
    return [
        # a viewer at the smallest resolution: launches, latency and the blocking read
        dict(name="still_512x256_d8", path="still", kind=1, depth=8, w=512, h=256),
        # the flagship flight: terrain and spheres, every image delivered
        dict(name="clip_warp_1920x1024_d11", path="clip", mode="warp", kind=2, depth=11, w=1920, h=1024, frames=8),
        # the same program in a window of no special size
        dict(name="clip_warp_1361x763_d10", path="clip", mode="warp", kind=2, depth=10, w=1361, h=763, frames=8),
        # fast flight through a cave: many holes, divergent short rays
        dict(name="clip_cave_1280x720_d10", path="clip", mode="warp", kind=4, depth=10, w=1280, h=720, frames=8),
        # every frame raycast in full (reference quality, training targets)
        dict(name="clip_full_1920x1024_d11", path="clip", mode="full", kind=2, depth=11, w=1920, h=1024, frames=2),
        # the flagship flight with the learned hole filler
        dict(name="clip_learned_1920x1024_d11", path="clip", mode="learned", kind=2, depth=11, w=1920, h=1024,
             frames=4),
        # a host loop written for the reference, call by call
        dict(name="stages_1280x720_d10", path="stages", kind=2, depth=10, w=1280, h=720),
        # a render server: ten cameras of uneven size in one batch
        dict(name="batch_10_d10", path="batch", kind=2, depth=10, views=10, first=0),
        # the warp as a building block of another program
        dict(name="proj_1920x1024", path="proj", w=1920, h=1024),
        # training the filler on the small workload
        dict(name="train_512x256_d8", path="train", kind=1, depth=8, w=512, h=256, crops=16, crop=64, steps=4),
        # gradients for a trainer of the caller's own
        dict(name="grads_16x64", path="grads", crops=16, crop=64),
        # a scene edited while it is shown
        dict(name="scene_d9", path="scene", kind=2, depth=9, w=640, h=480),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def size(most):  # from a thumbnail to `most` pixels wide, odd widths among them
        w = log_int(160, most)
        return w, max(96, int(w * rng.uniform(0.45, 0.75)))

    path = rng.choice(("clip", "clip", "clip", "still", "stages", "batch", "proj", "train", "grads", "scene"))
    if path == "clip":
        kind = rng.choice((1, 2, 2, 4))
        w, h = size(1920)
        return dict(path=path, mode=rng.choice(("warp", "warp", "full", "learned")), kind=kind,
                    depth=rng.choice(DEPTHS[kind]), w=w, h=min(h, 1024), frames=rng.randint(1, 4))
    if path in ("still", "stages"):
        kind = rng.choice((1, 2, 4))
        w, h = size(1280)
        return dict(path=path, kind=kind, depth=rng.choice([d for d in DEPTHS[kind] if d <= 10]), w=w, h=h)
    if path == "batch":
        return dict(path=path, kind=2, depth=rng.choice((9, 10)), views=rng.randint(2, 8), first=rng.randint(0, 3))
    if path == "proj":
        w, h = size(1920)
        return dict(path=path, w=w, h=min(h, 1024))
    if path == "train":
        w, h = size(768)
        return dict(path=path, kind=1, depth=rng.choice(DEPTHS[1]), w=w, h=h, crops=log_int(2, 32),
                    crop=8 * rng.randint(3, 8), steps=rng.randint(1, 3))
    if path == "grads":
        return dict(path=path, crops=log_int(1, 24), crop=8 * rng.randint(2, 8))
    w, h = size(800)
    return dict(path="scene", kind=rng.choice((1, 2)), depth=9, w=w, h=h)


# ---------------------------------------------------------------- assets and flights
@functools.lru_cache(maxsize=8)
def scene_words(kind, depth):
    """(words, root) of the shared scene: a program loads it once."""
    make = S.scene_gpu if kind == 4 else S.scene
    args = () if kind == 4 else (SPHERES.get((kind, depth), 0),)
    xyz, rgba = make(kind, 1000 + kind, depth, *args)
    return S.build_octree_gpu(xyz, rgba, depth)


SPHERES = {(2, 9): 200, (2, 10): 1000, (2, 11): 2000}


def flight(kind, depth, seed, frames=PATH_FRAMES):
    """FrameParams of a seeded flight, scaled from the workloads' motion."""
    s = 2.0 ** depth
    vox, yaw, height, pitch = {1: (2.0, 0.5, 0.94 * s, 0.35), 2: (8.0 * s / 2048, 1.0, 0.68 * s, 0.30),
                               4: (32.0 * s / 4096, 5.0, 0.5 * s, 0.05)}[kind]
    rows = S.camera_path(3000 + seed, depth, frames, vox, yaw, height, pitch)
    out = []
    for row in rows:
        a = [float(v) for v in row]
        out.append(S.camera(a[0], a[1], a[2], a[3:6], depth, 0)[0])
    return out


def next_params(s):
    """The next camera of the state's flight, with the running frame counter."""
    n, k = s["frame"], len(s["flight"])
    t = n % (2 * k - 2)
    p = s["flight"][t if t < k else 2 * k - 2 - t]
    p.frame = n
    s["frame"] = n + 1
    return p


def context(kind, depth, w, h):
    words, root = scene_words(kind, depth)
    c = S.Context(0)
    c.upload_octree(words, root, depth)
    c.resize(w, h)
    return c


def pinned(w, h):
    return torch.empty((h, w), dtype=torch.int32, pin_memory=True)


def as_words(t):
    return t.numpy().view(np.uint32)


def filler():
    cnn = S.Cnn(0)
    learned.load(cnn)
    return cnn


# ---------------------------------------------------------------- prepare
def prepare(case, seed):
    return {"clip": prepare_clip, "still": prepare_clip, "stages": prepare_clip, "batch": prepare_batch,
            "proj": prepare_proj, "train": prepare_train, "grads": prepare_grads,
            "scene": prepare_scene}[case["path"]](case, seed)


def render(s, c, p):
    mode = s["mode"]
    if mode == "full":
        c.frame_full(p)
    elif mode == "learned":
        c.frame_warp_learned(s["cnn"], p)
    else:
        c.frame_warp(p)


def prepare_clip(case, seed):
    w, h = case["w"], case["h"]
    s = dict(case=case, mode=case.get("mode", "warp"), frame=0, flight=flight(case["kind"], case["depth"], seed),
             ctx=context(case["kind"], case["depth"], w, h), images=[])
    if s["mode"] == "learned":
        s["cnn"] = filler()
    if case["path"] == "clip":
        s["images"] = [pinned(w, h) for _ in range(case["frames"])]
    for _ in range(WARM_FRAMES):
        render(s, s["ctx"], next_params(s))
    s["ctx"].sync()
    return s


def view_sizes(case):
    return [VIEWS[(case["first"] + i) % len(VIEWS)] for i in range(case["views"])]


def prepare_batch(case, seed):
    rng = np.random.default_rng(seed)
    n = case["views"]
    res = view_sizes(case)  # the same mix for every seed
    s = dict(case=case, cnn=filler(), views=[], images=[pinned(*r) for r in res],
             ctxs=[context(case["kind"], case["depth"], *r) for r in res])
    s["batch"] = S.Batch(s["ctxs"])
    for _ in range(n):
        s["views"].append(dict(frame=0, flight=flight(case["kind"], case["depth"], int(rng.integers(1 << 20)))))
    for _ in range(WARM_FRAMES):
        s["batch"].frame_warp_learned(s["cnn"], [next_params(v) for v in s["views"]])
    s["batch"].sync()
    return s


def prepare_proj(case, seed):
    """A cached frame as the caller's device tensors: plane 2 holds the words
    and world positions of a rendered frame, the others are empty."""
    w, h = case["w"], case["h"]
    path = flight(1, 9, seed, 8)
    c = context(1, 9, w, h)
    c.frame_full(path[0])
    c.sync()
    words = np.full((4, h, w), S.HOLE, np.uint32)
    coords = np.zeros((4, h, w, 4), np.float32)
    words[2], coords[2] = c.screen(0), c.coords(0)
    c.close()
    return dict(case=case, p=path[3], screen=torch.from_numpy(words.view(np.int32)).cuda(),
                coords=torch.from_numpy(coords).cuda())


def prepare_train(case, seed):
    w, h = case["w"], case["h"]
    s = dict(case=case, cnn=S.Cnn(0, seed=1 + seed % 1000), frame=0, step=0,
             flight=flight(case["kind"], case["depth"], seed), warp=context(case["kind"], case["depth"], w, h),
             full=context(case["kind"], case["depth"], w, h))
    for _ in range(WARM_FRAMES):
        p = next_params(s)
        s["warp"].frame_warp_learned(None, p, 256)
        s["full"].frame_full(p)
    s["warp"].sync()
    s["full"].sync()
    return s


def bf16_bits(x):
    return torch.from_numpy(np.ascontiguousarray(x, np.float32)).to(torch.bfloat16).view(torch.int16).numpy().view(
        np.uint16)


def grads_inputs(case, seed):
    """Crops as the filler sees them: smooth colours and depth, hole blobs,
    targets near the colours, the loss on the holes."""
    rng = np.random.default_rng(seed)
    b, n = case["crops"], case["crop"]
    coarse = rng.random((b, n // 8 + 1, n // 8 + 1, 4), np.float32).repeat(8, 1).repeat(8, 2)[:, :n, :n]
    smooth = 0.9 * coarse + 0.1 * rng.random((b, n, n, 4), np.float32)
    hole = rng.random((b, n // 2, n // 2), np.float32).repeat(2, 1).repeat(2, 2) < 0.2
    x = np.zeros((b, n, n, 16), np.float32)
    x[..., :4] = np.where(hole[..., None], 0.0, smooth)
    x[..., 4] = hole
    return bf16_bits(x), np.ascontiguousarray(smooth[..., :3]), hole.astype(np.float32)


def prepare_grads(case, seed):
    return dict(case=case, cnn=filler(), inputs=grads_inputs(case, seed))


@functools.lru_cache(maxsize=4)
def voxel_stream(kind, depth):
    return S.scene(kind, 1000 + kind, depth, SPHERES.get((kind, depth), 0))


def prepare_scene(case, seed):
    """The shared voxel stream with a seeded tenth of its voxels repainted."""
    kind, depth = case["kind"], case["depth"]
    xyz, rgba = voxel_stream(kind, depth)
    pick = np.random.default_rng(seed).random(len(rgba), np.float32)
    return dict(case=case, ctx=context(kind, depth, case["w"], case["h"]), p=flight(kind, depth, seed, 2)[0],
                xyz=xyz, rgba=np.where(pick < 0.1, rgba ^ np.uint32(0x58), rgba))


# ---------------------------------------------------------------- run
def run(s):
    return {"clip": run_clip, "still": run_still, "stages": run_stages, "batch": run_batch, "proj": run_proj,
            "train": run_train, "grads": run_grads, "scene": run_scene}[s["case"]["path"]](s)


def run_clip(s):
    out = []
    for image in s["images"]:
        render(s, s["ctx"], next_params(s))
        words = as_words(image)
        s["ctx"].read_image_async(words)
        out.append(words)
    return out


def run_still(s):
    render(s, s["ctx"], next_params(s))
    return s["ctx"].image()


def run_stages(s):
    c, p = s["ctx"], next_params(s)
    c.memset(0, S.HOLE, 4 * c.N)
    c.proj(1, p)
    c.proj(2, p)
    c.counthole()
    c.sumids()
    c.writeids()
    c.raycast_holes(p)
    c.raycast_rect(p, *S.tile_schedule(c.res_x, c.res_y, p.frame))
    c.copy_cache(2)
    c.fillhole()
    c.colorize()
    return c.image()


def run_batch(s):
    s["batch"].frame_warp_learned(s["cnn"], [next_params(v) for v in s["views"]])
    s["batch"].sync()
    out = [as_words(i) for i in s["images"]]
    for c, words in zip(s["ctxs"], out):
        c.read_image_async(words)
    return out


def run_proj(s):
    w, h = s["case"]["w"], s["case"]["h"]
    s["screen"][0].fill_(S.HOLE - (1 << 32))
    S.proj_noalloc(0, s["screen"].data_ptr(), s["coords"].data_ptr(), w, h, 2, s["p"],
                   torch.cuda.current_stream().cuda_stream)
    return s["screen"][0], s["coords"][0]


def run_train(s):
    case = s["case"]
    for _ in range(case["steps"]):
        p = next_params(s)
        s["warp"].frame_warp_learned(None, p, 256)
        s["full"].frame_full(p)
        s["cnn"].train_step(s["warp"], s["full"], p, case["crops"], case["crop"], seed=s["step"], lr=1e-3)
        s["step"] += 1
    return s["cnn"].params()


def run_grads(s):
    grads, loss = s["cnn"].gradients(*s["inputs"])
    return grads, np.float32(loss)


def run_scene(s):
    words, root = S.build_octree_gpu(s["xyz"], s["rgba"], s["case"]["depth"])
    c = s["ctx"]
    c.upload_octree(words, root, s["case"]["depth"])
    c.frame_full(s["p"])
    return words, c.image()


# ---------------------------------------------------------------- work
CNN_FLOPS = 2 * 9 * (5 * 32 + 32 * 32 + 32 * 32 + 32 * 3)  # per output pixel of the four layers
RAY_FLOPS = 5000  # a primary ray: about 100 DDA steps of some 50 operations
WARP_FLOPS = 30   # a warped sample
HOLES = {1: 0.06, 2: 0.05, 4: 0.2}  # share of the pixels that the hole list traces in a warp frame


def frame_work(case, n):
    """Bytes and flops of one frame of n pixels.  A warp frame reads the
    cached plane (word and position), writes the new plane, its cached copy
    and the image; a full frame writes plane and image."""
    if case.get("mode") == "full":
        return 20 * n + 4 * n, n * RAY_FLOPS
    flops = n * WARP_FLOPS + n * (1 / 32 + HOLES[case["kind"]]) * RAY_FLOPS
    if case.get("mode") == "learned":
        flops += 0.05 * n * CNN_FLOPS
    return 20 * n + 20 * n + 20 * n + 4 * n, flops


def work(case):
    path = case["path"]
    n = case.get("w", 0) * case.get("h", 0)
    if path in ("clip", "still", "stages"):
        b, f = frame_work(case, n)
        k = case.get("frames", 1)
        return dict(bytes=k * b, flops=k * f)
    if path == "batch":
        n = sum(w * h for w, h in view_sizes(case))
        b, f = frame_work(dict(case, mode="learned"), n)
        return dict(bytes=b, flops=f)
    if path == "proj":
        return dict(bytes=20 * n + 20 * n, flops=n * WARP_FLOPS)
    if path == "train":
        pix = case["crops"] * case["crop"] ** 2
        b, f = frame_work(dict(case, mode="warp"), n)
        b2, f2 = frame_work(dict(case, mode="full"), n)
        return dict(bytes=case["steps"] * (b + b2 + 24 * pix), flops=case["steps"] * (f + f2 + 3 * pix * CNN_FLOPS))
    if path == "grads":
        pix = case["crops"] * case["crop"] ** 2
        return dict(bytes=pix * (32 + 16) + 4 * 27760, flops=3 * pix * CNN_FLOPS)
    voxels = {1: 850000, 2: 3800000}[case["kind"]]
    return dict(bytes=voxels * 10 + 4 * 4000000 * 3 + 24 * n, flops=n * RAY_FLOPS)


# ---------------------------------------------------------------- exact
def exact(case, seed):
    """Gradients and loss in 64 bits; the other paths return words, bytes or
    positions of hits that have no value apart from the traversal's own
    arithmetic, and the trained parameters of a run of steps."""
    if case["path"] != "grads":
        return None
    x, target, mask = grads_inputs(case, seed)
    flat = np.load(learned.WEIGHTS, allow_pickle=False)["params"].astype(np.float64)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    a = torch.from_numpy(x.view(np.int16)).view(torch.bfloat16).to(torch.float64).permute(0, 3, 1, 2).to(dev)
    shapes, leaves, ofs = ((16, 32), (32, 32), (32, 32), (32, 16)), [], 0
    for layer, (cin, cout) in enumerate(shapes):
        n = 9 * cin * cout
        wt = torch.from_numpy(flat[ofs:ofs + n].reshape(9, cout, cin)).to(dev).requires_grad_()
        bias = torch.from_numpy(flat[ofs + n:ofs + n + cout]).to(dev).requires_grad_()
        ofs += n + cout
        leaves += [wt, bias]
        # the convolution as nine shifted products: plain matrix products in 64 bits
        h, w = a.shape[2:]
        pad = torch.nn.functional.pad(a, (1, 1, 1, 1)).permute(0, 2, 3, 1)
        y = bias
        for t in range(9):
            y = y + pad[:, t // 3:t // 3 + h, t % 3:t % 3 + w, :].reshape(-1, cin) @ wt[t].t()
        y = y.reshape(-1, h, w, cout).permute(0, 3, 1, 2)
        a = y if layer == 3 else torch.relu(y)
    rgb = a[:, :3].permute(0, 2, 3, 1)
    m = torch.from_numpy(mask.astype(np.float64)).to(dev)
    d = rgb - torch.from_numpy(target.astype(np.float64)).to(dev)
    loss = (m[..., None] * d * d).sum() / (3 * m.sum())
    loss.backward()
    grads = torch.cat([v.grad.reshape(-1) for v in leaves]).cpu().numpy()
    return grads, float(loss.detach())
