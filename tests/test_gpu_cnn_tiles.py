"""The fused tile kernel at the edges of its work split: fewer tiles than
workgroups, exactly two per compute unit's worth, one more, several rounds;
all 16 input channels in use; crops that reach over every screen edge."""
import numpy as np
import pytest

import cnn_ref as R
import svo_amd as S
from svo_amd import learned as L
from svo_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [1, 2, 511, 512, 513, 1300])
def test_tiles_by_count(count):
    """Every tile equals, bit for bit, the same tile in a call of its own, and
    the FP64 network within the bound of the fused forward (5e-3 relative to
    the norm: bf16 activations, FP32 sums)."""
    rng = np.random.default_rng(count)
    c = S.Cnn(0, seed=3)
    try:
        x = rng.uniform(0, 1, (count, 24, 24, 16)).astype(np.float32)
        bits = R.bf16_bits(x)
        out = c.forward_tiles(bits)
        for i in sorted({0, count // 2, count - 1}):
            assert np.array_equal(out[i], c.forward_tiles(bits[i:i + 1])[0]), i
            ref, _ = R.forward(c.params().astype(np.float64), R.bits_to_f64(bits[i:i + 1]))
            d = out[i] - ref[0, 4:20, 4:20, :3]
            assert np.linalg.norm(d) < 5e-3 * np.linalg.norm(ref[0, 4:20, 4:20, :3]), i
    finally:
        c.close()


@pytest.mark.parametrize("res", [(37, 21), (130, 67), (16, 16)])
def test_frame_tiles_at_screen_edges(res):
    """Learned frames at sizes whose last tiles are cut by the screen: the
    tile kernel against the per-layer kernels (same bounds as at the full
    size: 4 levels, 0.5 on average)."""
    name = "flythrough_256"
    words, root, depth, _ = W.octree(name)
    rows = W.path(name, 8)
    cnn = S.Cnn(0)
    L.load(cnn, L.WEIGHTS)
    a, b = S.Context(0), S.Context(0)
    try:
        for c in (a, b):
            c.upload_octree(words, root, depth)
            c.resize(*res)
        n_cnn = 0
        for f in range(8):
            p = W.frame_params(name, rows, f)
            for c, fused in ((a, True), (b, False)):
                cnn.set_fused(fused)
                c.frame_warp_learned(cnn, p, 256)
                c.sync()
            assert np.array_equal(a.screen(), b.screen()), f
            holes = (a.screen(2) == 0xFFFFFF00).reshape(-1)
            ia, ib = (c.image().reshape(-1, 1).view(np.uint8).astype(int) for c in (a, b))
            assert np.array_equal(ia[~holes], ib[~holes]), f
            n_cnn += int(holes.sum())
            if holes.any():
                d = np.abs(ia - ib)[holes]
                assert d.max() <= 4 and d.mean() < 0.5, (f, d.max(), d.mean())
        assert n_cnn > 0
    finally:
        a.close()
        b.close()
        cnn.close()
