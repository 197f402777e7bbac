"""The gradient kernels at the edges of their split: crops with fewer pixels
than slices, slices that end inside a group of steps, crops of one row of
tiles, more crops than are made together."""
import numpy as np
import pytest

import cnn_ref as R
import svo_amd as S

pytestmark = pytest.mark.gpu


def batch(rng, B, H, W):
    x = np.zeros((B, H, W, 16), np.float32)
    x[..., :5] = rng.uniform(0, 1, (B, H, W, 5))
    return (R.bf16_bits(x), rng.uniform(0, 1, (B, H, W, 3)).astype(np.float32),
            (rng.random((B, H, W)) < 0.4).astype(np.float32))


@pytest.mark.parametrize("shape", [(1, 8, 8), (1, 16, 16), (2, 8, 24), (3, 16, 24), (2, 24, 40), (1, 8, 136), (4, 56, 8)])
def test_gradients_by_shape(shape):
    """Every layer's weights and biases against the FP64 network, within the
    bounds of the other gradient test (3e-2 relative to a layer's norm: the
    backward keeps dZ in bf16; the loss 1e-3)."""
    rng = np.random.default_rng(shape[0] * 1000 + shape[2])
    bits, target, mask = batch(rng, *shape)
    c = S.Cnn(0, seed=9)
    try:
        g, loss = c.gradients(bits, target, mask)
        p = c.params().astype(np.float64)
        x = R.bits_to_f64(bits)
        ref_loss, ref = R.loss_and_grads(p, x, target.astype(np.float64), mask.astype(np.float64))
        assert abs(loss - ref_loss) <= 1e-3 * abs(ref_loss)
        o = 0
        for ci, co in zip(R.CIN, R.COUT):
            for n in (9 * ci * co, co):
                d = np.linalg.norm(g[o:o + n] - ref[o:o + n])
                assert d <= 3e-2 * np.linalg.norm(ref[o:o + n]) + 1e-12, (o, n, d)
                o += n
    finally:
        c.close()


def test_many_crops_equal_few():
    """2,500 crops (their gradients are made layer by layer) of which only the
    first ten carry loss: the other crops' partials are zeros, so the gradients
    equal those of the ten crops alone (made in one launch) bit for bit."""
    rng = np.random.default_rng(5)
    bits, target, mask = batch(rng, 2500, 8, 8)
    mask[10:] = 0
    c = S.Cnn(0, seed=9)
    try:
        few, loss_few = c.gradients(bits[:10], target[:10], mask[:10])
        many, loss_many = c.gradients(bits, target, mask)
        assert np.array_equal(few, many)
        assert abs(loss_few - loss_many) <= 1e-5 * abs(loss_few)
    finally:
        c.close()
