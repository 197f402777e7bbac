"""Device memory the network holds: a forward takes the activations only, the
gradients' buffers come with the first gradients, and neither grows again for
batches that fit."""
import ctypes as C

import numpy as np
import pytest

import svo_amd as S

pytestmark = pytest.mark.gpu

SLACK = 32 << 20  # allocations are rounded up; streams and code objects


def free_bytes():
    hip = C.CDLL("libamdhip64.so.7")
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def test_workspace_per_pixel():
    B, H, W = 16, 256, 256
    pix = B * H * W
    x = np.zeros((B, H, W, 16), np.uint16)
    c = S.Cnn(0, seed=9)
    try:
        c.forward(x[:1, :8, :8])
        before = free_bytes()
        c.forward(x)
        forward = before - free_bytes()
        print("forward", forward / pix, "bytes per pixel", flush=True)
        assert forward <= 288 * pix + SLACK
        c.gradients(x, np.zeros((B, H, W, 3), np.float32), np.ones((B, H, W), np.float32))
        both = before - free_bytes()
        print("and gradients", both / pix, flush=True)
        assert both <= 528 * pix + B * 108 * 1024 + 2 * pix + SLACK
        c.forward(x[:8])
        c.gradients(x[:3], np.zeros((3, H, W, 3), np.float32), np.ones((3, H, W), np.float32))
        assert before - free_bytes() <= both + SLACK
    finally:
        c.close()


def test_gradients_after_a_larger_forward():
    """The two workspaces grow on their own: gradients of a batch smaller and
    larger than the forward's before it, against a network that made nothing
    else."""
    rng = np.random.default_rng(3)
    x = rng.integers(0, 0x3F80, (5, 24, 24, 16)).astype(np.uint16)
    x[..., 5:] = 0
    target = rng.random((5, 24, 24, 3)).astype(np.float32)
    mask = (rng.random((5, 24, 24)) < 0.5).astype(np.float32)
    c = S.Cnn(0, seed=4)
    try:
        c.forward(x[:3])
        for n in (2, 5, 1):
            other = S.Cnn(0, seed=4)
            try:
                got, want = c.gradients(x[:n], target[:n], mask[:n])[0], other.gradients(x[:n], target[:n], mask[:n])[0]
                assert np.array_equal(got, want), n
                assert np.array_equal(c.forward(x[:n]), other.forward(x[:n])), n
            finally:
                other.close()
    finally:
        c.close()
